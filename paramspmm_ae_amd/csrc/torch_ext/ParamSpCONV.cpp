// Python module `ParamSpCONV`: the fused GCN layer ops of the reference's SpCONV/SpCONV.cpp:496-512
// (glue in SpCONV/SpCONV.h:43-193): forward A*(H*W), backward [ (A*dY)*W^T, H^T*(A*dY) ]; and this build's layers and losses as
// autograd nodes.  The sparse products and, for widths that are multiples of 16 up to 128 and 1024 rows or more, the dense
// ones are libparamsp_hip.so's (but see kept_order_is_ours); torch::mm forms the others.
#include "glue_common.h"
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/saved_variable.h>

using namespace pspglue;
using torch::Tensor;

static void check_cf(int CF, int fmt = 0)
{
    if (fmt == 4) {  // windowed csr: CF names the kernel variant
        TORCH_CHECK(CF >= 0 && CF <= 3, "the windowed format takes variant 0..3 in place of CF");
        return;
    }
    // SpCONV dispatches CF 1..4 only (SpCONV/SpCONV.cpp:92-124)
    TORCH_CHECK((CF >= 1 && CF <= 8) || (CF & PSP_CF_NATIVE), "CF must be 1..8 (or a native configuration)");
}

// A*D for a dense D, result cut back to rows(D) (the blocked formats compute into an even-padded buffer,
// SpCONV/SpCONV.h:115-118)
static Tensor aggregate(int fmt, const Tensor &D, const Tensor &rowPtr, const Tensor &colIdx, const Tensor &values,
                        const Tensor *target_row, int CF, int blkWarpNum)
{
    check_cf(CF, fmt);
    Tensor Dc = D.contiguous();
    Tensor Y = spmm_new(fmt, Dc, rowPtr, colIdx, values, target_row, CF, blkWarpNum);
    if (Y.size(0) != Dc.size(0)) Y = Y.narrow(0, 0, Dc.size(0));
    return Y;
}

// Rows from which the library's dense kernels are used (PyTorch's GEMM below): they cost one launch with the activation
// or the mask folded in, where PyTorch needs one for each.  us at 1024 rows against PyTorch, relu(Z) W, masked X W^T and weight
// gradient: 48 x 48 5 / 25, 5 / 27, 10 / 26; 96 x 96 12 / 25, 12 / 27, 20 / 26; 128 x 128 18 / 25, 19 / 27, 13 / 26.  What PyTorch
// takes is its launches, so the line could lie lower; fewer rows have not been measured.
constexpr long kDenseRows = 1024;

// Where a product's result is the activation of a ReLU network (GCN, GIN), another order of its sum puts some element on the
// other side of zero, which drops or adds a whole term of the gradient: a training run would not repeat the figures it gave
// before.  Those products stay with the order that each shape has always had: the library's (ascending k up to 32 columns,
// see dense_xw.hip) at the shapes below from 16384 rows on, PyTorch's GEMM elsewhere.  This is a list of what was the library's
// before its kernel took every width, not a line that was measured: at the shapes it leaves to PyTorch the kernel is the faster
// one (48 x 48, 10^6 rows: 81 us against 208).  Gradients (X W^T and the weight gradient) and the attention layer have no such
// step behind them and take the library's kernel at every shape.
enum class Order { any, kept };
static bool kept_order_is_ours(long n, long K1, long K2)
{
    const bool pow2 = K1 == 16 || K1 == 32 || K1 == 64 || K1 == 128;
    return n >= 16384 && (K2 <= 32 ? K1 <= 64 || (K1 == 128 && K2 == 16) : (K2 == 64 || K2 == 128) && pow2);
}

// Weight gradients leave their kernels as partial products of the workgroups.  The sums of everything one backward call forms
// share a launch (psp_sum_partials_f32): flush() before the gradients are handed out.  What a launch less saves, some 5 us,
// counts where the workspaces are small; past kHeldBytes they are summed and given back at once (64 MB a layer at 128 x 128).
struct PartialSums {
    static constexpr size_t kHeldBytes = (size_t)32 << 20;
    std::vector<psp_partial_sum> jobs;
    std::vector<Tensor> held;  // workspaces and results, until the launch
    size_t held_bytes = 0;
    psp_stream_t stream = nullptr;
    void add(const Tensor &ws, Tensor &dW, int count)
    {
        jobs.push_back({fp(ws), fpw(dW), count, (int)dW.numel()});
        held.push_back(ws);
        held.push_back(dW);
        held_bytes += ws.nbytes();
        stream = stream_of(ws);
        if (held_bytes > kHeldBytes) flush();
    }
    void flush()
    {
        if (jobs.empty()) return;
        DeviceGuard guard(held[0].device());
        ok(psp_sum_partials_f32(jobs.data(), (int)jobs.size(), stream));
        jobs.clear();
        held.clear();
        held_bytes = 0;
    }
};
static int ok_count(int rc)
{
    ok(rc);
    return rc;
}

// The rows of a dense kernel's operand.  Those kernels read 16 bytes at a time and their entry points refuse other starts; a
// contiguous view into a flat buffer may start on any element and is copied.
static Tensor rows16(const Tensor &t)
{
    Tensor c = t.contiguous();
    return (reinterpret_cast<uintptr_t>(c.const_data_ptr()) & 15) == 0 ? c : c.clone();
}

// H^T * AG.  For narrow layers the product is a reduction over ~10^6 rows into a tiny matrix, which the library
// streams at memory speed; everything else goes to torch::mm.
static Tensor weight_gradient(const Tensor &H, const Tensor &AG, PartialSums *sums = nullptr, bool relu = false)
{
    const bool narrow = H.dim() == 2 && AG.dim() == 2 && H.size(0) == AG.size(0) && H.size(0) >= kDenseRows &&
                        H.scalar_type() == torch::kFloat32 && AG.scalar_type() == torch::kFloat32 &&
                        psp_gemm_atb_supported((int)H.size(1), (int)AG.size(1));
    if (!narrow) return torch::mm((relu ? torch::relu(H) : H).t(), AG);
    Tensor Hc = rows16(H), Gc = rows16(AG);
    DeviceGuard guard(Hc.device());
    Tensor dW = torch::empty({Hc.size(1), Gc.size(1)}, Hc.options());
    // partial products of the workgroups go through a workspace and are added in a fixed order (no atomics)
    const long long ws_floats = psp_gemm_atb_workspace_floats(Hc.size(0), (int)Hc.size(1), (int)Gc.size(1));
    Tensor ws = torch::empty({(long)ws_floats}, Hc.options());
    const int count = ok_count(psp_gemm_atb_ws_act_f32(fp(Hc), fp(Gc), sums ? nullptr : fpw(dW), Hc.size(0), (int)Hc.size(1),
                                                       (int)Gc.size(1), relu ? 1 : 0, fpw(ws), ws_floats, stream_of(Hc)));
    if (sums) sums->add(ws, dW, count);
    return dW;
}

// X * W (or X * W^T): the library's kernel for narrow layers on many rows, torch::mm otherwise
static Tensor dense_xw(const Tensor &X, const Tensor &W, bool transW, Order order)
{
    const long K1 = X.dim() == 2 ? X.size(1) : -1;
    const bool shapes = X.dim() == 2 && W.dim() == 2 && W.size(transW ? 1 : 0) == K1;
    const long K2 = shapes ? W.size(transW ? 0 : 1) : -1;
    const bool narrow = shapes && X.size(0) >= kDenseRows && X.scalar_type() == torch::kFloat32 &&
                        W.scalar_type() == torch::kFloat32 && X.is_cuda() && W.is_cuda() &&
                        psp_gemm_xw_supported((int)K1, (int)K2) && (order == Order::any || kept_order_is_ours(X.size(0), K1, K2));
    if (!narrow) return torch::mm(X, transW ? W.t() : W);
    Tensor Xc = rows16(X), Wc = W.contiguous();
    DeviceGuard guard(Xc.device());
    Tensor Y = torch::empty({Xc.size(0), K2}, Xc.options());
    ok(psp_gemm_xw_f32(fp(Xc), fp(Wc), fpw(Y), Xc.size(0), (int)K1, (int)K2, transW ? 1 : 0, stream_of(Xc)));
    return Y;
}

// The same two products with the ReLU between two layers folded in (psp_gemm_xw_act_f32 / psp_gemm_atb_ws_act_f32);
// shapes the library does not cover apply the activation with PyTorch and multiply with torch::mm.
static Tensor dense_relu_xw(const Tensor &Z, const Tensor &W, Order order)
{
    const long K1 = Z.dim() == 2 ? Z.size(1) : -1;
    const bool shapes = Z.dim() == 2 && W.dim() == 2 && W.size(0) == K1;
    const bool narrow = shapes && Z.size(0) >= kDenseRows && Z.scalar_type() == torch::kFloat32 && W.scalar_type() == torch::kFloat32 &&
                        psp_gemm_xw_supported((int)K1, (int)W.size(1)) &&
                        (order == Order::any || kept_order_is_ours(Z.size(0), K1, W.size(1)));
    if (!narrow) return torch::mm(torch::relu(Z), W);
    Tensor Zc = rows16(Z), Wc = W.contiguous();
    DeviceGuard guard(Zc.device());
    Tensor Y = torch::empty({Zc.size(0), Wc.size(1)}, Zc.options());
    ok(psp_gemm_xw_act_f32(fp(Zc), fp(Wc), fpw(Y), Zc.size(0), (int)K1, (int)Wc.size(1), 0, 1, nullptr, stream_of(Zc)));
    return Y;
}
// (AG * W^T) where Z > 0, else 0
static Tensor dense_xwt_masked(const Tensor &AG, const Tensor &W, const Tensor &Z)
{
    const long K1 = AG.dim() == 2 ? AG.size(1) : -1;
    const bool shapes = AG.dim() == 2 && W.dim() == 2 && W.size(1) == K1 && Z.dim() == 2 && Z.size(0) == AG.size(0) &&
                        Z.size(1) == W.size(0);
    const bool narrow = shapes && AG.size(0) >= kDenseRows && AG.scalar_type() == torch::kFloat32 && W.scalar_type() == torch::kFloat32 &&
                        Z.scalar_type() == torch::kFloat32 && psp_gemm_xw_supported((int)K1, (int)W.size(0));
    if (!narrow) return at::threshold_backward(torch::mm(AG, W.t()), Z, 0);  // what F.relu's backward runs
    Tensor Gc = rows16(AG), Wc = W.contiguous(), Zc = rows16(Z);
    DeviceGuard guard(Gc.device());
    Tensor Y = torch::empty({Gc.size(0), Wc.size(0)}, Gc.options());
    ok(psp_gemm_xw_act_f32(fp(Gc), fp(Wc), fpw(Y), Gc.size(0), (int)K1, (int)Wc.size(0), 1, 0, fp(Zc), stream_of(Gc)));
    return Y;
}
// relu(Z)^T * AG
static Tensor weight_gradient_relu(const Tensor &Z, const Tensor &AG, PartialSums *sums = nullptr)
{
    return weight_gradient(Z, AG, sums, true);
}
// {(AG * W^T) where Z > 0, relu(Z)^T * AG}: one launch where the library has the pair (psp_dense_grad_f32)
static std::pair<Tensor, Tensor> dense_grads_relu(const Tensor &AG, const Tensor &W, const Tensor &Z, PartialSums *sums)
{
    const bool pair = AG.dim() == 2 && W.dim() == 2 && Z.dim() == 2 && Z.size(0) == AG.size(0) && Z.size(1) == W.size(0) &&
                      AG.size(1) == W.size(1) && AG.size(0) >= kDenseRows && AG.scalar_type() == torch::kFloat32 &&
                      W.scalar_type() == torch::kFloat32 && Z.scalar_type() == torch::kFloat32 &&
                      psp_dense_grad_supported((int)W.size(0), (int)W.size(1));
    if (!pair) return {dense_xwt_masked(AG, W, Z), weight_gradient_relu(Z, AG, sums)};
    Tensor Gc = rows16(AG), Wc = W.contiguous(), Zc = rows16(Z);
    DeviceGuard guard(Gc.device());
    const int K1 = (int)Wc.size(0), K2 = (int)Wc.size(1);
    Tensor dZ = torch::empty_like(Zc), dW = torch::empty_like(Wc);
    const long long ws_floats = psp_dense_grad_workspace_floats(Gc.size(0), K1, K2);
    Tensor ws = torch::empty({(long)ws_floats}, Gc.options());
    const int count = ok_count(psp_dense_grad_f32(fp(Gc), fp(Zc), fp(Wc), fpw(dZ), sums ? nullptr : fpw(dW), Gc.size(0), K1, K2, fpw(ws),
                                                  ws_floats, stream_of(Gc)));
    if (sums) sums->add(ws, dW, count);
    return {dZ, dW};
}

// GCN layer that reads its input through a ReLU: A * (relu(Z) * W).  fmt: 0 csr, 1 csr_split, 2 bcsr, 3 bcsr_split.
// No counterpart among the reference's bindings: its driver applies F.relu between the layers as a pass of its own
// (GNN.py:43-61); the algebra of the layer itself is SpCONV/SpCONV.h:43-71.
static Tensor relu_input_forward(int fmt, Tensor Z, Tensor W, Tensor rowPtr, Tensor colIdx, Tensor values,
                                 c10::optional<Tensor> target_row, int CF, int bw)
{
    need_gpu(Z, "input");
    need_gpu(W, "weight");
    TORCH_CHECK(fmt >= 0 && fmt <= 4 && (fmt == 1 || fmt == 3) == target_row.has_value(), "format code and target_row disagree");
    return aggregate(fmt, dense_relu_xw(Z, W, Order::kept), rowPtr, colIdx, values, target_row ? &*target_row : nullptr, CF, bw);
}
// [dZ, dW] = [ ((A dY) W^T) where Z > 0,  relu(Z)^T (A dY) ]
static std::vector<Tensor> relu_input_backward(int fmt, Tensor dY, Tensor Z, Tensor W, Tensor rowPtr, Tensor colIdx,
                                               Tensor values, c10::optional<Tensor> target_row, int CF, int bw)
{
    need_gpu(Z, "input");
    need_gpu(W, "weight");
    TORCH_CHECK(fmt >= 0 && fmt <= 4 && (fmt == 1 || fmt == 3) == target_row.has_value(), "format code and target_row disagree");
    Tensor AG = aggregate(fmt, dY, rowPtr, colIdx, values, target_row ? &*target_row : nullptr, CF, bw);
    auto r = dense_grads_relu(AG, W, Z, nullptr);
    return {r.first, r.second};
}

// A * D alone, for callers that place the sparse product on the narrower side of the layer: (A H) W costs a sparse
// product of width in_features where A (H W) costs one of width out_features.  No counterpart among the reference's
// bindings, whose layer is always A (H W) (SpCONV/SpCONV.h:43-48).
static Tensor aggregate_op(int fmt, Tensor D, Tensor rowPtr, Tensor colIdx, Tensor values, c10::optional<Tensor> target_row,
                           int CF, int bw)
{
    need_gpu(D, "input");
    TORCH_CHECK(fmt >= 0 && fmt <= 4 && (fmt == 1 || fmt == 3) == target_row.has_value(), "format code and target_row disagree");
    return aggregate(fmt, D, rowPtr, colIdx, values, target_row ? &*target_row : nullptr, CF, bw);
}

// A * max(D, 0) and / or (A * D) kept where mask > 0: the ReLU between two layers folded into the sparse product
// (psp_spmm_act_f32).  Used by the layers that aggregate first (GIN: (A X) W): the activation is applied as the rows of
// D are gathered, its backward as the rows of the gradient are written.  No counterpart among the reference's
// bindings: its driver runs F.relu as a pass of its own (GNN.py:63-78).  float64 and mask shapes the kernel does not
// take fall back to PyTorch's passes around the plain product.
static Tensor aggregate_act_op(int fmt, Tensor D, Tensor rowPtr, Tensor colIdx, Tensor values, c10::optional<Tensor> target_row,
                               int CF, int bw, bool relu_input, c10::optional<Tensor> mask)
{
    need_gpu(D, "input");
    TORCH_CHECK(fmt >= 0 && fmt <= 4 && (fmt == 1 || fmt == 3) == target_row.has_value(), "format code and target_row disagree");
    check_cf(CF, fmt);
    const Tensor *tr = target_row ? &*target_row : nullptr;
    if (mask) {
        need_gpu(*mask, "mask");
        TORCH_CHECK(mask->dim() == 2 && mask->size(0) == D.size(0) && mask->size(1) == D.size(1), "mask must have the shape of the result");
    }
    const bool blocked = pspglue::fmt_blocked(fmt);
    const bool fused = D.scalar_type() == torch::kFloat32 && (!mask || mask->scalar_type() == torch::kFloat32) &&
                       D.size(1) > 0 && D.size(0) > 0 && (!blocked || D.size(0) % 2 == 0 || !mask);
    if (!fused) {
        Tensor Y = aggregate(fmt, relu_input ? torch::relu(D) : D, rowPtr, colIdx, values, tr, CF, bw);
        return mask ? at::threshold_backward(Y, *mask, 0) : Y;
    }
    Tensor Dc = D.contiguous();
    check_spmm_args(fmt, Dc, rowPtr, colIdx, values, tr);
    DeviceGuard guard(Dc.device());
    const long rows_out = blocked ? (Dc.size(0) + 1) / 2 * 2 : Dc.size(0);
    Tensor Mc;
    if (mask) Mc = mask->contiguous();
    Tensor Y = torch::empty({rows_out, Dc.size(1)}, Dc.options());
    if (fmt == 4)  // windowed csr: the activation is applied as the window is staged, the mask where a row is stored
        ok(psp_spmm_window_f32(ip(rowPtr), ip(colIdx), fp(values), fp(Dc), fpw(Y), pspglue::fmt_rows(fmt, rowPtr),
                               (int)colIdx.size(0), (int)Dc.size(1), (int)rows_out, CF, relu_input ? 1 : 0,
                               mask ? fp(Mc) : nullptr, stream_of(Dc)));
    else
        ok(psp_spmm_act_f32(fmt, ip(rowPtr), ip(colIdx), fp(values), tr ? ip(*tr) : nullptr, fp(Dc), fpw(Y),
                            (int)rowPtr.size(0) - 1, (int)Dc.size(1), (int)rows_out, CF, bw, relu_input ? 1 : 0,
                            mask ? fp(Mc) : nullptr, stream_of(Dc)));
    if (Y.size(0) != Dc.size(0)) Y = Y.narrow(0, 0, Dc.size(0));
    return Y;
}

// Windowed layout, square layer of 16 or 32 columns: the dense product folded into the sparse one
// (psp_spmm_window_xw_f32).  Returns [Y] or [Y, A f(X)]:  Y = ((A f(X)) W | W^T), kept where mask > 0 when a mask is given.
static bool window_xw_supported(long N) { return N == 16 || N == 32; }
static std::vector<Tensor> window_xw(Tensor X, Tensor W, bool transW, Tensor rowPtr_w, Tensor colIdx_w, Tensor values_w,
                                     bool relu_input, c10::optional<Tensor> mask, bool want_raw)
{
    need_gpu(X, "input");
    need_gpu(W, "weight");
    Tensor Xc = X.contiguous(), Wc = W.contiguous();
    check_spmm_args(4, Xc, rowPtr_w, colIdx_w, values_w, nullptr);
    need_f32(Wc, "weight", 2);
    const long N = Xc.size(1);
    TORCH_CHECK(window_xw_supported(N) && Wc.size(0) == N && Wc.size(1) == N,
                "window_xw: a square weight matrix of 16 or 32 columns, as wide as the input");
    pspglue::same_device(Xc, Wc, "window_xw");
    Tensor Mc;
    if (mask) {
        need_gpu(*mask, "mask");
        TORCH_CHECK(mask->scalar_type() == torch::kFloat32 && mask->dim() == 2 && mask->size(0) == Xc.size(0) && mask->size(1) == N,
                    "mask must be float32 with the shape of the result");
        Mc = mask->contiguous();
    }
    DeviceGuard guard(Xc.device());
    Tensor Y = torch::empty_like(Xc), R;
    if (want_raw) R = torch::empty_like(Xc);
    ok(psp_spmm_window_xw_f32(ip(rowPtr_w), ip(colIdx_w), fp(values_w), fp(Xc), fp(Wc), transW ? 1 : 0, fpw(Y),
                              want_raw ? fpw(R) : nullptr, pspglue::fmt_rows(4, rowPtr_w), (int)colIdx_w.size(0), (int)N,
                              (int)Xc.size(0), relu_input ? 1 : 0, mask ? fp(Mc) : nullptr, stream_of(Xc)));
    if (want_raw) return {Y, R};
    return {Y};
}

// Backward on the windowed layout with the weight gradient formed in the sparse kernel (psp_spmm_window_grad_f32): dW = f(Z)^T (A G)
// and, with W, dZ = ((A G) W^T) where Z > 0, else A G when want_ag.  Returns {dW (whole after sums.flush()), dZ or A G or nothing}.
static bool window_grad_supported(const Tensor &G, const Tensor &Z, bool dense)
{
    return G.dim() == 2 && Z.dim() == 2 && G.size(0) == Z.size(0) && G.scalar_type() == torch::kFloat32 && Z.scalar_type() == torch::kFloat32 &&
           psp_spmm_window_grad_supported((int)G.size(1), (int)Z.size(1), dense ? 1 : 0);
}
static std::vector<Tensor> window_grad(Tensor G, Tensor Z, bool relu_z, const Tensor *W, bool want_ag, Tensor rowPtr_w, Tensor colIdx_w,
                                       Tensor values_w, PartialSums &sums)
{
    Tensor Gc = rows16(G), Zc = rows16(Z), Wc;
    check_spmm_args(4, Gc, rowPtr_w, colIdx_w, values_w, nullptr);
    pspglue::same_device(Gc, Zc, "window_grad");
    if (W) {
        Wc = W->contiguous();
        need_f32(Wc, "weight", 2);
        pspglue::same_device(Gc, Wc, "window_grad");
    }
    DeviceGuard guard(Gc.device());
    const int M = pspglue::fmt_rows(4, rowPtr_w), N = (int)Gc.size(1), KZ = (int)Zc.size(1);
    TORCH_CHECK(Gc.size(0) >= M && Zc.size(0) >= M && (!W || (Wc.size(0) == KZ && Wc.size(1) == N)), "window_grad: shapes");
    const long long ws_floats = psp_spmm_window_grad_workspace_floats(M, N, KZ, W ? 1 : 0);
    Tensor dW = torch::empty({KZ, N}, Gc.options()), ws = torch::empty({(long)ws_floats}, Gc.options()), Y;
    if (W || want_ag) Y = torch::empty_like(Gc);
    const int count = ok_count(psp_spmm_window_grad_f32(ip(rowPtr_w), ip(colIdx_w), fp(values_w), fp(Gc), fp(Zc), KZ, relu_z ? 1 : 0,
                                                        W ? fp(Wc) : nullptr, Y.defined() ? fpw(Y) : nullptr, nullptr, fpw(ws), ws_floats,
                                                        M, (int)colIdx_w.size(0), N, (int)Gc.size(0), stream_of(Gc)));
    sums.add(ws, dW, count);
    return {dW, Y};
}

// ---- attention layer on the windowed layout: SDDMM and SpMM of a direction in one launch ---------------------------------
static bool attn_window_supported(long K) { return K >= 4 && K % 4 == 0 && K <= PSP_ATTN_WINDOW_MAX_K; }

static void check_attn_window(const Tensor &X, const Tensor &rowPtr_w, const Tensor &colIdx_w, const char *what)
{
    need_gpu(X, what);
    need_gpu(rowPtr_w, "rowPtr_w");
    need_gpu(colIdx_w, "colIdx_w");
    need_f32(X, what, 2);
    need_i32(rowPtr_w, "rowPtr_w");
    need_i32(colIdx_w, "colIdx_w");
    pspglue::same_device(X, rowPtr_w, "attn_window");
    pspglue::same_device(X, colIdx_w, "attn_window");
    TORCH_CHECK(rowPtr_w.size(0) >= 2 && rowPtr_w.size(0) % 2 == 0, "rowPtr of the windowed format has 2 M + 2 entries");
    TORCH_CHECK(attn_window_supported(X.size(1)), "attn_window: the width must be a multiple of 4 up to ", PSP_ATTN_WINDOW_MAX_K);
    TORCH_CHECK((rowPtr_w.size(0) - 2) / 2 <= X.size(0), "rowPtr_w describes more rows than the dense operand has");
}

// (X, rowPtr_w, colIdx_w, alpha | None) -> [att = alpha <X_i, X_j> per stored entry, Y = att-weighted sum of the X rows]
static std::vector<Tensor> attn_window_forward(Tensor X, Tensor rowPtr_w, Tensor colIdx_w, c10::optional<Tensor> alpha)
{
    check_attn_window(X, rowPtr_w, colIdx_w, "X");
    if (alpha) {
        need_gpu(*alpha, "alpha");
        TORCH_CHECK(alpha->scalar_type() == torch::kFloat32 && alpha->numel() == 1, "alpha is one float32 on the device");
        pspglue::same_device(X, *alpha, "attn_window");
    }
    pspglue::DeviceGuard guard(X.device());
    Tensor att = torch::empty({colIdx_w.size(0)}, X.options());
    Tensor Y = torch::empty_like(X);
    const float *a = alpha ? alpha->data_ptr<float>() : nullptr;
    ok(psp_attn_window_forward_f32(ip(rowPtr_w), ip(colIdx_w), fp(X), a, colIdx_w.numel() ? fpw(att) : nullptr, fpw(Y),
                                   (int)(rowPtr_w.size(0) - 2) / 2, (int)colIdx_w.size(0), (int)X.size(1), (int)X.size(0),
                                   stream_of(X)));
    return {att, Y};
}

// (dY, att, rowPtr_w, colIdx_w) -> [G = att-weighted sum of the dY rows, sum_p <dY_i, dY_j> float(col(p)) as a 1-element tensor]
static std::vector<Tensor> attn_window_backward(Tensor dY, Tensor att, Tensor rowPtr_w, Tensor colIdx_w)
{
    check_attn_window(dY, rowPtr_w, colIdx_w, "dY");
    need_gpu(att, "att");
    need_f32(att, "att", 1);
    TORCH_CHECK(att.size(0) == colIdx_w.size(0), "att has one value per stored entry");
    pspglue::same_device(dY, att, "attn_window");
    pspglue::DeviceGuard guard(dY.device());
    Tensor G = torch::empty_like(dY);
    Tensor wsum = torch::empty({1}, dY.options());
    ok(psp_attn_window_backward_f32(ip(rowPtr_w), ip(colIdx_w), att.numel() ? fp(att) : nullptr, fp(dY), fpw(G), wsum.data_ptr<float>(),
                                    (int)(rowPtr_w.size(0) - 2) / 2, (int)colIdx_w.size(0), (int)dY.size(1), (int)dY.size(0),
                                    stream_of(dY)));
    return {G, wsum};
}

// ---- the same on the PCSR formats (fmt 0..3) ---------------------------------------------------------------------------
static bool attn_supported(long K) { return K >= 4 && K <= PSP_ATTN_MAX_K; }

static void check_attn(int fmt, const Tensor &X, const Tensor &rowPtr, const Tensor &colIdx, const Tensor &values,
                       const Tensor *target_row, int blkWarpNum)
{
    TORCH_CHECK(fmt >= 0 && fmt <= 3 && (fmt == 1 || fmt == 3) == (target_row != nullptr), "format code and target_row disagree");
    check_spmm_args(fmt, X, rowPtr, colIdx, values, target_row);
    TORCH_CHECK(X.scalar_type() == torch::kFloat32 && attn_supported(X.size(1)), "attn: float32 rows of 4 to ", PSP_ATTN_MAX_K, " columns");
    TORCH_CHECK((blkWarpNum & ~PSP_BW_STRIPE_MASK) == 4 || (blkWarpNum & ~PSP_BW_STRIPE_MASK) == 8, "blkWarpNum must be 4 or 8");
    // the kernel reads both rows of a block-row
    if (fmt == 2) TORCH_CHECK(2 * (rowPtr.size(0) - 1) <= X.size(0), "the dense operand needs two rows per block-row (pad it to an even row count)");
    if (fmt == 3) TORCH_CHECK(X.size(0) % 2 == 0, "the dense operand needs two rows per block-row (pad it to an even row count)");
}

// (fmt, X, rowPtr, colIdx, values, target_row | None, alpha | None, blkWarpNum) -> [att in the format's entry order, Y]
static std::vector<Tensor> attn_forward(int fmt, Tensor X, Tensor rowPtr, Tensor colIdx, Tensor values, c10::optional<Tensor> target_row,
                                        c10::optional<Tensor> alpha, int blkWarpNum)
{
    const Tensor *tr = target_row ? &*target_row : nullptr;
    check_attn(fmt, X, rowPtr, colIdx, values, tr, blkWarpNum);
    if (alpha) {
        need_gpu(*alpha, "alpha");
        TORCH_CHECK(alpha->scalar_type() == torch::kFloat32 && alpha->numel() == 1, "alpha is one float32 on the device");
        pspglue::same_device(X, *alpha, "attn");
    }
    DeviceGuard guard(X.device());
    Tensor att = torch::empty_like(values), Y = torch::empty_like(X);
    ok(psp_attn_forward_f32(fmt, ip(rowPtr), ip(colIdx), fmt >= 2 ? fp(values) : nullptr, tr ? ip(*tr) : nullptr, fp(X),
                            alpha ? alpha->data_ptr<float>() : nullptr, fpw(att), fpw(Y), (int)rowPtr.size(0) - 1, (int)X.size(1),
                            (int)X.size(0), blkWarpNum, stream_of(X)));
    return {att, Y};
}

// (fmt, dY, att, rowPtr, colIdx, target_row | None, slot | None, blkWarpNum) -> [G, weight-gradient sum as a 1-element tensor];
// slot: what each score's dot product is multiplied with (CSR: None for the entry's own column)
static std::vector<Tensor> attn_backward(int fmt, Tensor dY, Tensor att, Tensor rowPtr, Tensor colIdx, c10::optional<Tensor> target_row,
                                         c10::optional<Tensor> slot, int blkWarpNum)
{
    const Tensor *tr = target_row ? &*target_row : nullptr;
    TORCH_CHECK(fmt < 2 || slot.has_value(), "attn: 2x1 blocks take the columns of their slots");
    if (slot) {
        need_gpu(*slot, "slot");
        TORCH_CHECK(slot->scalar_type() == torch::kFloat32 && slot->numel() == att.numel(), "attn: slot has one float32 per score");
        pspglue::same_device(dY, *slot, "attn");
    }
    check_attn(fmt, dY, rowPtr, colIdx, att, tr, blkWarpNum);
    DeviceGuard guard(dY.device());
    const int nrows = (int)rowPtr.size(0) - 1, K = (int)dY.size(1);
    Tensor G = torch::empty_like(dY), wsum = torch::empty({1}, dY.options());
    Tensor ws = torch::empty({(long)psp_attn_workspace_floats(nrows, K)}, dY.options());
    ok(psp_attn_backward_f32(fmt, ip(rowPtr), ip(colIdx), fp(att), tr ? ip(*tr) : nullptr, slot ? fp(*slot) : nullptr, fp(dY), fpw(G), wsum.data_ptr<float>(),
                             fpw(ws), nrows, K, (int)dY.size(0), blkWarpNum, stream_of(dY)));
    return {G, wsum};
}

static Tensor forward_impl(int fmt, const Tensor &H, const Tensor &W, const Tensor &rowPtr, const Tensor &colIdx,
                           const Tensor &values, const Tensor *target_row, int CF, int blkWarpNum)
{
    need_gpu(H, "input");
    need_gpu(W, "weight");
    return aggregate(fmt, dense_xw(H, W, false, Order::kept), rowPtr, colIdx, values, target_row, CF, blkWarpNum);
}

static std::vector<Tensor> backward_impl(int fmt, const Tensor &dY, const Tensor &H, const Tensor &W, const Tensor &rowPtr,
                                         const Tensor &colIdx, const Tensor &values, const Tensor *target_row, int CF,
                                         int blkWarpNum)
{
    need_gpu(H, "H");
    need_gpu(W, "weight");
    // the reference multiplies by A, not A^T (SpCONV/SpCONV.h:67-71): exact for the symmetric matrices its
    // loaders build
    Tensor AG = aggregate(fmt, dY, rowPtr, colIdx, values, target_row, CF, blkWarpNum);
    return {dense_xw(AG, W, true, Order::any), weight_gradient(H, AG)};
}

// ---- mean NLL loss of the training step (an addition of this build; F.nll_loss in GNN.py:131-146) ----------
static void check_loss_args(const Tensor &logp, const Tensor &labels)
{
    need_gpu(logp, "log-probabilities");
    need_gpu(labels, "labels");
    TORCH_CHECK(logp.dim() == 2 && logp.scalar_type() == torch::kFloat32 && logp.is_contiguous(),
                "nll_loss_mean: log-probabilities must be a contiguous float32 [n, C] tensor");
    TORCH_CHECK(labels.dim() == 1 && labels.scalar_type() == torch::kInt64 && labels.is_contiguous() &&
                    labels.size(0) == logp.size(0),
                "nll_loss_mean: labels must be a contiguous int64 tensor with one entry per row");
    TORCH_CHECK(logp.device() == labels.device(), "nll_loss_mean: tensors on different devices");
}
// returns [loss (0-dim), stats (sum, count, stray labels, workspace) for the backward call]
static std::vector<Tensor> nll_loss_mean(Tensor logp, Tensor labels)
{
    check_loss_args(logp, labels);
    DeviceGuard guard(logp.device());
    Tensor loss = torch::empty({}, logp.options()), stats = torch::empty({(long)psp_nll_loss_stats_floats()}, logp.options());
    ok(psp_nll_loss_mean_f32(fp(logp), (const long long *)labels.data_ptr<int64_t>(), logp.size(0), (int)logp.size(1),
                             loss.data_ptr<float>(), stats.data_ptr<float>(), stream_of(logp)));
    return {loss, stats};
}
static Tensor nll_loss_mean_backward(Tensor labels, Tensor grad_loss, Tensor stats, long n, long C)
{
    need_gpu(labels, "labels");
    need_gpu(grad_loss, "grad_loss");
    need_gpu(stats, "stats");
    TORCH_CHECK(labels.scalar_type() == torch::kInt64 && labels.is_contiguous() && labels.numel() == n, "bad labels");
    TORCH_CHECK(grad_loss.scalar_type() == torch::kFloat32 && grad_loss.numel() == 1, "grad_loss must hold one float");
    TORCH_CHECK(stats.scalar_type() == torch::kFloat32 && stats.numel() >= 2 && stats.is_contiguous(), "bad stats");
    DeviceGuard guard(labels.device());
    Tensor grad = torch::empty({n, C}, stats.options());
    ok(psp_nll_loss_mean_backward_f32((const long long *)labels.data_ptr<int64_t>(), grad_loss.data_ptr<float>(),
                                      stats.data_ptr<float>(), n, (int)C, fpw(grad), stream_of(labels)));
    return grad;
}

// the same loss from the logits (log-softmax folded in): [loss, stats]; and its gradient w.r.t. the logits
static bool softmax_nll_supported(long C) { return psp_softmax_nll_supported((int)C) != 0; }
static std::vector<Tensor> softmax_nll_mean(Tensor logits, Tensor labels)
{
    check_loss_args(logits, labels);
    TORCH_CHECK(softmax_nll_supported(logits.size(1)), "softmax_nll_mean: the class count must be a multiple of 4 up to 64");
    DeviceGuard guard(logits.device());
    Tensor loss = torch::empty({}, logits.options()), stats = torch::empty({(long)psp_nll_loss_stats_floats()}, logits.options());
    ok(psp_softmax_nll_mean_f32(fp(logits), (const long long *)labels.data_ptr<int64_t>(), logits.size(0), (int)logits.size(1),
                                loss.data_ptr<float>(), stats.data_ptr<float>(), stream_of(logits)));
    return {loss, stats};
}
static Tensor softmax_nll_mean_backward(Tensor logits, Tensor labels, Tensor grad_loss, Tensor stats)
{
    check_loss_args(logits, labels);
    need_gpu(grad_loss, "grad_loss");
    need_gpu(stats, "stats");
    TORCH_CHECK(grad_loss.scalar_type() == torch::kFloat32 && grad_loss.numel() == 1, "grad_loss must hold one float");
    TORCH_CHECK(stats.scalar_type() == torch::kFloat32 && stats.numel() >= 2 && stats.is_contiguous(), "bad stats");
    DeviceGuard guard(logits.device());
    Tensor grad = torch::empty_like(logits);
    ok(psp_softmax_nll_mean_backward_f32(fp(logits), (const long long *)labels.data_ptr<int64_t>(), grad_loss.data_ptr<float>(),
                                         stats.data_ptr<float>(), logits.size(0), (int)logits.size(1), fpw(grad), stream_of(logits)));
    return grad;
}

// ---- the layers as autograd nodes ----------------------------------------------------------------------------------------
// One call from Python per layer and direction-free backward: the engine runs apply() without entering the interpreter.  As
// Python autograd Functions the five layers and the loss of a training step cost some 25 us each of interpreter and binding
// time, which on a graph of 20 K nodes was more than the GPU needs for the step (305 us per step, GPU busy 185).
struct Operator {  // what a layer needs of a pcsr_spmm
    int fmt;       // 0 csr, 1 csr_split, 2 bcsr, 3 bcsr_split, 4 windowed csr
    Tensor rowPtr, colIdx, val;
    c10::optional<Tensor> target_row;
    int CF, bw;
    bool fold_dense;      // windowed csr: fold a square dense product into the sparse kernel where there is one
    c10::optional<Tensor> slot;  // attention weight gradient: a column per score, where it is not the entry's own
    const Tensor *tr() const { return target_row ? &*target_row : nullptr; }
};
typedef std::shared_ptr<Operator> op_t;

using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

struct LayerNode : torch::autograd::Node {
    op_t op;
    SavedVariable a_, w_, z_;
    void release_variables() override
    {
        a_.reset_data();
        w_.reset_data();
        z_.reset_data();
    }
    Tensor a() { return a_.unpack(shared_from_this()); }
    Tensor w() { return w_.unpack(shared_from_this()); }
    Tensor z() { return z_.unpack(shared_from_this()); }
    bool wants(size_t i) { return task_should_compute_output(i); }
};

// The nodes have no forward-mode derivative.  What runs inside with_node is out of autograd's sight, so a tangent would be
// dropped, which says that the derivative is zero: refused as an autograd.Function without a jvp refuses it.
static void refuse_tangents(at::ArrayRef<Tensor> inputs)
{
    for (const Tensor &t : inputs)
        TORCH_CHECK_NOT_IMPLEMENTED(!t._fw_grad(0).defined(), "ParamSpCONV: the layers and losses have no forward-mode derivative");
}

// the result of `forward` (run without recording), with a node of type N behind it when an input asks for gradients
template <class N, class F> static Tensor with_node(const op_t &op, at::ArrayRef<Tensor> inputs, F forward)
{
    refuse_tangents(inputs);
    const bool record = torch::GradMode::is_enabled() &&
                        std::any_of(inputs.begin(), inputs.end(), [](const Tensor &t) { return t.requires_grad(); });
    std::shared_ptr<N> node;
    if (record) {
        node = std::shared_ptr<N>(new N(), torch::autograd::deleteNode);
        torch::autograd::edge_list edges;
        for (const Tensor &t : inputs) edges.push_back(torch::autograd::impl::gradient_edge(t));
        node->set_next_edges(std::move(edges));
        node->op = op;
    }
    Tensor out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        out = forward(node.get());
    }
    if (record) torch::autograd::set_history(out, node);
    return out;
}

static bool folds_dense(const Operator &o, const Tensor &Z, const Tensor &W)
{
    return o.fmt == 4 && o.fold_dense && W.size(0) == W.size(1) && W.size(0) == Z.size(1) && window_xw_supported(Z.size(1)) &&
           Z.scalar_type() == torch::kFloat32;
}

// The layers without attention, each direction once: for nodes of their own and for a whole network's.
enum Layer {
    kGCN = 0,             // A (H W); dH = (A dY) W^T, dW = H^T (A dY) -- A is symmetric (gnn_conv.py:13-107)
    kAggregateFirst = 1,  // (A H) W with A H kept: dW = (A H)^T dY, dH = A (dY W^T) -- the layer that widens its input, and
                          // GIN's (gnn_conv.py:202-220)
    kGCNReLU = 2,         // A (relu(Z) W): dZ = ((A dY) W^T) where Z > 0, dW = relu(Z)^T (A dY)
    kGINReLU = 3          // (A relu(Z)) W for a layer that widens its input: the activation is applied as the sparse product
                          // gathers the rows of Z, the gradient masked in a pass that follows the backward product
};
// kept: what the backward needs besides the input and the weights (A H; undefined for the kinds that keep nothing)
static Tensor layer_forward(int kind, const Operator &o, const Tensor &in, const Tensor &W, Tensor &kept)
{
    need_gpu(in, "input");
    need_gpu(W, "weight");
    switch (kind) {
    case kGCN: return aggregate(o.fmt, dense_xw(in, W, false, Order::kept), o.rowPtr, o.colIdx, o.val, o.tr(), o.CF, o.bw);
    case kAggregateFirst:
        kept = aggregate(o.fmt, in, o.rowPtr, o.colIdx, o.val, o.tr(), o.CF, o.bw);
        return dense_xw(kept, W, false, Order::kept);
    case kGCNReLU:
        // windowed layout, square layer: (A relu(Z)) W in one launch, the dense product in the kernel's epilogue
        if (folds_dense(o, in, W)) return window_xw(in, W, false, o.rowPtr, o.colIdx, o.val, true, c10::nullopt, false)[0];
        return relu_input_forward(o.fmt, in, W, o.rowPtr, o.colIdx, o.val, o.target_row, o.CF, o.bw);
    default:
        kept = aggregate_act_op(o.fmt, in, o.rowPtr, o.colIdx, o.val, o.target_row, o.CF, o.bw, true, c10::nullopt);
        return dense_xw(kept, W, false, Order::kept);
    }
}
// {gradient of the input, of the weights (whole after sums.flush())}, either undefined when not wanted; `in` may be undefined
// for kAggregateFirst
static std::pair<Tensor, Tensor> layer_backward(int kind, const Operator &o, const Tensor &g, const Tensor &in, const Tensor &W,
                                                const Tensor &kept, bool want_in, bool want_w, PartialSums &sums)
{
    Tensor dY = g.contiguous(), dIn, dW;
    if (kind == kGCN || kind == kGCNReLU) {
        const bool relu = kind == kGCNReLU;
        if (relu && folds_dense(o, in, W)) {
            // one launch delivers ((A dY) W^T) where Z > 0 (the input gradient) and the weight gradient
            auto r = window_grad(dY, in, true, &W, false, o.rowPtr, o.colIdx, o.val, sums);
            return {r[1], r[0]};
        }
        Tensor AG;
        if (o.fmt == 4 && want_w && window_grad_supported(dY, in, false)) {
            auto r = window_grad(dY, in, relu, nullptr, want_in, o.rowPtr, o.colIdx, o.val, sums);
            dW = r[0], AG = r[1];
        } else {
            AG = aggregate(o.fmt, dY, o.rowPtr, o.colIdx, o.val, o.tr(), o.CF, o.bw);
            if (relu && want_in && want_w) return dense_grads_relu(AG, W, in, &sums);
            if (want_w) dW = weight_gradient(in, AG, &sums, relu);
        }
        if (want_in) dIn = relu ? dense_xwt_masked(AG, W, in) : dense_xw(AG, W, true, Order::any);
        return {dIn, dW};
    }
    if (want_in) {
        Tensor D = dense_xw(dY, W, true, Order::any);
        dIn = kind == kGINReLU ? aggregate_act_op(o.fmt, D, o.rowPtr, o.colIdx, o.val, o.target_row, o.CF, o.bw, false, in)
                               : aggregate(o.fmt, D, o.rowPtr, o.colIdx, o.val, o.tr(), o.CF, o.bw);
    }
    if (want_w) dW = weight_gradient(kept, dY, &sums);
    return {dIn, dW};
}

template <int KIND> struct PlainLayer : LayerNode {  // a_ = input (kAggregateFirst: none), z_ = kept
    variable_list apply(variable_list &&g) override
    {
        if (!g[0].defined()) return {Tensor(), Tensor()};
        constexpr bool in = KIND != kAggregateFirst, keeps = KIND == kAggregateFirst || KIND == kGINReLU;
        PartialSums sums;
        auto r = layer_backward(KIND, *op, g[0], in ? a() : Tensor(), w(), keeps ? z() : Tensor(), wants(0), wants(1), sums);
        sums.flush();
        return {r.first, r.second};
    }
};
struct GCNFunction : PlainLayer<kGCN> {};
struct GCNAggregateFirstFunction : PlainLayer<kAggregateFirst> {};
struct GCNReLUInputFunction : PlainLayer<kGCNReLU> {};
struct GINFunction : PlainLayer<kAggregateFirst> {};
struct GINReLUInputFunction : PlainLayer<kGINReLU> {};
template <class N, int KIND> static Tensor plain_layer(op_t op, Tensor H, Tensor W)
{
    return with_node<N>(op, {H, W}, [&](N *n) {
        Tensor kept, out = layer_forward(KIND, *op, H, W, kept);
        if (n) {
            if (KIND != kAggregateFirst) n->a_ = SavedVariable(H, false);
            n->w_ = SavedVariable(W, false);
            if (kept.defined()) n->z_ = SavedVariable(kept, false);
        }
        return out;
    });
}

// The attention layer, its sparse work one launch per direction (gnn_conv.py:128-180): X' = f(X) W, att = alpha <X'_i, X'_j>,
// out = att-weighted sum of the X' rows; the gradients are the reference's literal formulas
static std::vector<Tensor> attn_fused_forward(const Operator &o, const Tensor &Xp, const Tensor &alpha)
{
    if (o.fmt == 4) return attn_window_forward(Xp, o.rowPtr, o.colIdx, alpha);
    return attn_forward(o.fmt, Xp, o.rowPtr, o.colIdx, o.val, o.target_row, alpha, o.bw);
}
struct AGNNFunction : LayerNode {  // a_ = X, z_ = att
    bool relu_input = false;
    std::vector<int64_t> alpha_shape;
    variable_list apply(variable_list &&g) override
    {
        if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
        Tensor X = a(), W = w(), att = z(), dY = g[0].contiguous();
        auto r = op->fmt == 4 ? attn_window_backward(dY, att, op->rowPtr, op->colIdx)
                              : attn_backward(op->fmt, dY, att, op->rowPtr, op->colIdx, op->target_row, op->slot, op->bw);
        Tensor dX, dW;
        if (relu_input && wants(0) && wants(1)) {
            std::tie(dX, dW) = dense_grads_relu(r[0], W, X, nullptr);
        } else {
            if (wants(0)) dX = relu_input ? dense_xwt_masked(r[0], W, X) : dense_xw(r[0], W, true, Order::any);
            if (wants(1)) dW = weight_gradient(X, r[0], nullptr, relu_input);
        }
        return {dX, dW, r[1].reshape({1, 1}).expand(alpha_shape)};
    }
};
static Tensor agnn_layer(op_t op, Tensor X, Tensor W, Tensor attention_w, bool relu_input)
{
    need_gpu(X, "input");
    need_gpu(W, "weight");
    return with_node<AGNNFunction>(op, {X, W, attention_w}, [&](AGNNFunction *n) {
        Tensor Xp = relu_input ? dense_relu_xw(X, W, Order::any) : dense_xw(X, W, false, Order::any);
        auto r = attn_fused_forward(*op, Xp, attention_w.reshape({-1}).narrow(0, 0, 1));
        if (n) {
            n->a_ = SavedVariable(X, false), n->w_ = SavedVariable(W, false), n->z_ = SavedVariable(r[0], false);
            n->relu_input = relu_input;
            n->alpha_shape = attention_w.sizes().vec();
        }
        return r[1];
    });
}

struct NllLossMean : LayerNode {  // a_ = labels, z_ = stats
    int64_t n = 0, C = 0;
    variable_list apply(variable_list &&g) override
    {
        if (!g[0].defined()) return {Tensor(), Tensor()};
        return {wants(0) ? nll_loss_mean_backward(a(), g[0].contiguous(), z(), n, C) : Tensor(), Tensor()};
    }
};
static Tensor nll_loss_layer(Tensor logp, Tensor labels)
{
    return with_node<NllLossMean>(nullptr, {logp, labels}, [&](NllLossMean *n) {
        auto r = nll_loss_mean(logp, labels);
        if (n) n->a_ = SavedVariable(labels, false), n->z_ = SavedVariable(r[1], false), n->n = logp.size(0), n->C = logp.size(1);
        return r[0];
    });
}
struct SoftmaxNllMean : LayerNode {  // a_ = labels, w_ = logits, z_ = stats
    variable_list apply(variable_list &&g) override
    {
        if (!g[0].defined()) return {Tensor(), Tensor()};
        return {wants(0) ? softmax_nll_mean_backward(w(), a(), g[0].contiguous(), z()) : Tensor(), Tensor()};
    }
};
static Tensor softmax_nll_layer(Tensor logits, Tensor labels)
{
    return with_node<SoftmaxNllMean>(nullptr, {logits, labels}, [&](SoftmaxNllMean *n) {
        auto r = softmax_nll_mean(logits, labels);
        if (n) n->a_ = SavedVariable(labels, false), n->w_ = SavedVariable(logits, false), n->z_ = SavedVariable(r[1], false);
        return r[0];
    });
}

// A training step's network and loss, nll_loss(log_softmax(layers(x)), labels), as one node.  On a graph of 20 K nodes the step is
// bound by the host: six nodes cost the engine some 80 us, and each layer's weight gradient a launch for its sum.  In a backward
// pass that does not keep the graph, what a layer saved is given back when its gradients are launched, as nodes of their own
// would do (10^6 rows, hidden 128: every layer's input or kept product is 512 MB).
struct NetworkLoss : LayerNode {  // a_ = labels, w_ = logits, z_ = stats
    struct Part {
        int kind;
        op_t op;
        SavedVariable in, w, kept;
        void release() { in.reset_data(), w.reset_data(), kept.reset_data(); }
    };
    std::vector<Part> parts;
    bool last_pass = false;
    void will_release_variables() override { last_pass = true; }
    void release_variables() override
    {
        LayerNode::release_variables();
        for (Part &p : parts) p.release();
    }
    variable_list apply(variable_list &&g) override
    {
        variable_list out(1 + parts.size());
        if (!g[0].defined()) return out;
        auto self = shared_from_this();
        size_t lowest = 0;  // the lowest input (x, then the weights) that asks for its gradient
        while (lowest < out.size() && !wants(lowest)) lowest++;
        if (lowest == out.size()) return out;
        Tensor d = softmax_nll_mean_backward(w(), a(), g[0].contiguous(), z());
        if (last_pass) LayerNode::release_variables();
        PartialSums sums;
        for (size_t l = parts.size(); l-- > 0 && lowest <= l + 1;) {
            Part &p = parts[l];
            const bool keeps = p.kind == kAggregateFirst || p.kind == kGINReLU;
            std::tie(d, out[l + 1]) = layer_backward(p.kind, *p.op, d, p.kind == kAggregateFirst ? Tensor() : p.in.unpack(self), p.w.unpack(self),
                                                     keeps ? p.kept.unpack(self) : Tensor(), lowest <= l, wants(l + 1), sums);
            if (last_pass) p.release();
            if (!wants(l + 1)) out[l + 1] = Tensor();
        }
        if (wants(0)) out[0] = d;
        sums.flush();
        return out;
    }
};
static Tensor network_loss(std::vector<int> kinds, std::vector<op_t> ops, Tensor x, std::vector<Tensor> weights, Tensor labels)
{
    const size_t L = weights.size();
    TORCH_CHECK(L > 0 && kinds.size() == L && ops.size() == L, "network_loss: one kind, operator and weight matrix per layer");
    for (int k : kinds) TORCH_CHECK(k >= kGCN && k <= kGINReLU, "network_loss: unknown kind of layer");
    std::vector<Tensor> inputs{x};
    inputs.insert(inputs.end(), weights.begin(), weights.end());
    return with_node<NetworkLoss>(nullptr, inputs, [&](NetworkLoss *n) {
        Tensor h = x;
        if (n) n->parts.reserve(L);
        for (size_t l = 0; l < L; l++) {
            Tensor kept, out = layer_forward(kinds[l], *ops[l], h, weights[l], kept);
            if (n) {
                n->parts.emplace_back();
                NetworkLoss::Part &p = n->parts.back();
                p.kind = kinds[l], p.op = ops[l];
                p.w = SavedVariable(weights[l], false);
                if (kinds[l] != kAggregateFirst) p.in = SavedVariable(h, false);
                if (kept.defined()) p.kept = SavedVariable(kept, false);
            }
            h = out;
        }
        auto r = softmax_nll_mean(h, labels);
        if (n) n->a_ = SavedVariable(labels, false), n->w_ = SavedVariable(h, false), n->z_ = SavedVariable(r[1], false);
        return r[0];
    });
}

// the nodes under their own names in Python (type(t.grad_fn).__name__)
template <class N> static void register_node(const char *name)
{
    static PyTypeObject type;
    torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
    torch::autograd::registerCppFunction(typeid(N), &type);
}

#define PSP_CONV(NAME, FMT)                                                                                       \
    static Tensor NAME##_forward(Tensor H, Tensor W, Tensor rowPtr, Tensor colIdx, Tensor values, int CF, int bw)  \
    {                                                                                                             \
        return forward_impl(FMT, H, W, rowPtr, colIdx, values, nullptr, CF, bw);                                  \
    }                                                                                                             \
    static std::vector<Tensor> NAME##_backward(Tensor dY, Tensor H, Tensor W, Tensor rowPtr, Tensor colIdx,       \
                                               Tensor values, int CF, int bw)                                     \
    {                                                                                                             \
        return backward_impl(FMT, dY, H, W, rowPtr, colIdx, values, nullptr, CF, bw);                             \
    }
#define PSP_CONV_SPLIT(NAME, FMT)                                                                                 \
    static Tensor NAME##_forward(Tensor H, Tensor W, Tensor rowPtr, Tensor colIdx, Tensor values, Tensor tr,      \
                                 int CF, int bw)                                                                  \
    {                                                                                                             \
        return forward_impl(FMT, H, W, rowPtr, colIdx, values, &tr, CF, bw);                                      \
    }                                                                                                             \
    static std::vector<Tensor> NAME##_backward(Tensor dY, Tensor H, Tensor W, Tensor rowPtr, Tensor colIdx,       \
                                               Tensor values, Tensor tr, int CF, int bw)                          \
    {                                                                                                             \
        return backward_impl(FMT, dY, H, W, rowPtr, colIdx, values, &tr, CF, bw);                                 \
    }

PSP_CONV(csr_spmm, 0)
PSP_CONV_SPLIT(csr_split_spmm, 1)
PSP_CONV(bcsr_spmm, 2)
PSP_CONV_SPLIT(bcsr_split_spmm, 3)

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    pspglue::check_abi();
    register_node<GCNFunction>("GCNFunctionBackward");
    register_node<GCNAggregateFirstFunction>("GCNAggregateFirstFunctionBackward");
    register_node<GCNReLUInputFunction>("GCNReLUInputFunctionBackward");
    register_node<GINFunction>("GINFunctionBackward");
    register_node<GINReLUInputFunction>("GINReLUInputFunctionBackward");
    register_node<AGNNFunction>("AGNNFunctionBackward");
    register_node<NllLossMean>("NllLossMeanBackward");
    register_node<SoftmaxNllMean>("SoftmaxNllMeanBackward");
    register_node<NetworkLoss>("NetworkLossBackward");
    py::class_<Operator, op_t>(m, "Operator", "what a layer needs of a pcsr_spmm")
        .def(py::init([](int fmt, Tensor rowPtr, Tensor colIdx, Tensor val, c10::optional<Tensor> target_row, int CF, int bw,
                         bool fold_dense, c10::optional<Tensor> slot) {
            TORCH_CHECK(fmt >= 0 && fmt <= 4 && (fmt == 1 || fmt == 3) == target_row.has_value(), "format code and target_row disagree");
            return std::make_shared<Operator>(Operator{fmt, rowPtr, colIdx, val, target_row, CF, bw, fold_dense, slot});
        }));
    m.def("gcn_layer", &plain_layer<GCNFunction, kGCN>, "A (H W): (operator, H, W)");
    m.def("gcn_aggregate_first_layer", &plain_layer<GCNAggregateFirstFunction, kAggregateFirst>, "(A H) W: (operator, H, W)");
    m.def("gcn_relu_layer", &plain_layer<GCNReLUInputFunction, kGCNReLU>, "A (relu(Z) W): (operator, Z, W)");
    m.def("gin_layer", &plain_layer<GINFunction, kAggregateFirst>, "(A X) W: (operator, X, W)");
    m.def("gin_relu_layer", &plain_layer<GINReLUInputFunction, kGINReLU>, "(A relu(Z)) W: (operator, Z, W)");
    m.def("agnn_layer", &agnn_layer, "attention layer: (operator, X, W, attention_w, relu_input)");
    m.def("nll_loss_layer", &nll_loss_layer, "mean negative log-likelihood: (log-probabilities, int64 labels)");
    m.def("softmax_nll_layer", &softmax_nll_layer, "nll_loss(log_softmax(logits), labels), mean over the rows");
    m.def("network_loss", &network_loss,
          "nll_loss(log_softmax(layers(x)), labels): (kinds 0 gcn, 1 aggregate first, 2 gcn of relu, 3 aggregate first of relu; operators, x, weights, labels)");
    m.def("split_csr", &pspglue::split_csr, "row split on the host");
    m.def("split_csr_par", &pspglue::split_csr_par, "row split on the host with a precomputed segment prefix");
    // addition of this build: H^T * G for tall-skinny operands (a kernel of the library's for multiples of 16 up to 128 and 1024
    // rows or more, else torch::mm)
    m.def("weight_gradient", [](Tensor H, Tensor G) {
        need_gpu(H, "H");
        need_gpu(G, "G");
        return weight_gradient(H, G);
    }, "H^T * G");
    m.def("dense_xw", [](Tensor X, Tensor W, bool transW) {
        need_gpu(X, "X");
        need_gpu(W, "W");
        return dense_xw(X, W, transW, transW ? Order::any : Order::kept);
    }, "X * W (transW false) or X * W^T for tall-skinny X: (X, W, transW)");
    // the dense products of a layer that reads its input through a ReLU, for layers that place them around their
    // own sparse operators (the attention layer): max(Z, 0) * W, (G * W^T) where Z > 0, max(Z, 0)^T * G
    m.def("dense_relu_xw", [](Tensor Z, Tensor W) {
        need_gpu(Z, "Z");
        need_gpu(W, "W");
        return dense_relu_xw(Z, W, Order::kept);
    }, "max(Z, 0) * W: (Z, W)");
    m.def("dense_xwt_masked", [](Tensor G, Tensor W, Tensor Z) {
        need_gpu(G, "G");
        need_gpu(W, "W");
        need_gpu(Z, "Z");
        return dense_xwt_masked(G, W, Z);
    }, "(G * W^T) where Z > 0, else 0: (G, W, Z)");
    m.def("weight_gradient_relu", [](Tensor Z, Tensor G) {
        need_gpu(Z, "Z");
        need_gpu(G, "G");
        return weight_gradient_relu(Z, G);
    }, "max(Z, 0)^T * G: (Z, G)");
    m.def("nll_loss_mean", &nll_loss_mean, "[loss, stats] of the mean negative log-likelihood (log-probabilities, int64 labels)");
    m.def("nll_loss_mean_backward", &nll_loss_mean_backward, "gradient w.r.t. the log-probabilities: (labels, grad_loss, stats, n, C)");
    m.def("softmax_nll_supported", &softmax_nll_supported, "is there a fused log-softmax + NLL kernel for this class count?");
    m.def("softmax_nll_mean", &softmax_nll_mean, "[loss, stats] of nll_loss(log_softmax(logits), labels), mean over the rows");
    m.def("softmax_nll_mean_backward", &softmax_nll_mean_backward, "gradient w.r.t. the logits: (logits, labels, grad_loss, stats)");
    m.def("attn_window_forward", &attn_window_forward,
          "attention layer on the windowed layout: (X, rowPtr_w, colIdx_w, alpha | None) -> [att, Y]");
    m.def("attn_window_backward", &attn_window_backward,
          "attention layer on the windowed layout: (dY, att, rowPtr_w, colIdx_w) -> [G, weight-gradient sum]");
    m.def("attn_window_supported", &attn_window_supported, "is there a fused attention kernel for this width?");
    m.def("attn_forward", &attn_forward,
          "attention layer on a PCSR format: (fmt 0..3, X, rowPtr, colIdx, values, target_row | None, alpha | None, blkWarpNum) -> [att, Y]");
    m.def("attn_backward", &attn_backward,
          "attention layer on a PCSR format: (fmt 0..3, dY, att, rowPtr, colIdx, target_row | None, slot | None, blkWarpNum) -> [G, weight-gradient sum]");
    m.def("attn_supported", &attn_supported, "is there a fused attention kernel for this width on the PCSR formats?");
    m.def("window_xw", &window_xw,
          "windowed layout, dense product folded in: (X, W, transW, rowPtr_w, colIdx_w, values_w, relu_input, mask | None, want_raw) -> [Y] or [Y, A f(X)]");
    m.def("window_xw_supported", &window_xw_supported, "widths the folded product exists for");
    m.def("aggregate", &aggregate_op, "A*D: (fmt, D, rowPtr, colIdx, values, target_row | None, CF, blkWarpNum)");
    m.def("aggregate_act", &aggregate_act_op,
          "A*max(D,0) (relu_input) and / or (A*D) where mask > 0: (fmt, D, rowPtr, colIdx, values, target_row | None, CF, blkWarpNum, relu_input, mask | None)");
    m.def("relu_input_forward", &relu_input_forward,
          "A*(relu(Z)*W): (fmt 0..3, Z, W, rowPtr, colIdx, values, target_row or None, CF, blkWarpNum)");
    m.def("relu_input_backward", &relu_input_backward,
          "[dZ, dW] of relu_input_forward: (fmt, dY, Z, W, rowPtr, colIdx, values, target_row or None, CF, blkWarpNum)");
    m.def("csr_spmm_forward", &csr_spmm_forward, "A*(H*W), CSR");
    m.def("csr_spmm_backward", &csr_spmm_backward, "[dH, dW], CSR");
    m.def("csr_split_spmm_forward", &csr_split_spmm_forward, "A*(H*W), row-split CSR");
    m.def("csr_split_spmm_backward", &csr_split_spmm_backward, "[dH, dW], row-split CSR");
    m.def("bcsr_spmm_forward", &bcsr_spmm_forward, "A*(H*W), 2x1 BCSR");
    m.def("bcsr_spmm_backward", &bcsr_spmm_backward, "[dH, dW], 2x1 BCSR");
    m.def("bcsr_split_spmm_forward", &bcsr_split_spmm_forward, "A*(H*W), row-split 2x1 BCSR");
    m.def("bcsr_split_spmm_backward", &bcsr_split_spmm_backward, "[dH, dW], row-split 2x1 BCSR");
}
