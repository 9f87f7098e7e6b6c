"""GCN / AGNN / GIN layers as autograd functions over the PCSR operators (same surface and the same forward /
backward algebra as the reference's gnn_conv.py:13-238).  The functions are nodes of ParamSpCONV: neither direction
enters the interpreter between two launches.  Layers look their operator up in ``spmm_dict`` by output width
(gnn_conv.py:121-124)."""
import math

import torch
from torch.nn.modules import module as _module

import paramspmm_ae_amd  # noqa: F401
import ParamSpCONV as SpCONV

n_heads = 1


def _bw(op):
    """blkWarpNum with the operator's launch flags (the XCD stripe chosen for its format, PCSR.pcsr_spmm.bw_flags)."""
    return op.blkWarpNum | getattr(op, "bw_flags", 0)


def _fmt(op):
    """Format code of the generic entry points (pcsr_spmm.fmt_code: 0 csr, 1 csr_split, 2 bcsr, 3 bcsr_split,
    4 windowed csr); operators of other origin are described by if_split / vec_size."""
    code = getattr(op, "fmt_code", None)
    return (1 if op.if_split else 0) + (2 if op.vec_size != 1 else 0) if code is None else code


def _row_ptr(op):
    return getattr(op, "spmm_rowPtr", op.rowPtr)


def _attn_fused(op, X, weights):
    """Does the attention layer's sparse work run as one launch per direction?  float32 rows of a width the fused kernels
    have, as many of them as the 2x1 blocks' rows need."""
    if X.dtype != torch.float32 or weights.dtype != torch.float32:
        return False
    width = int(weights.shape[1])
    if _fmt(op) == 4:
        return SpCONV.attn_window_supported(width)
    if op.vec_size not in (1, 2) or not SpCONV.attn_supported(width):
        return False
    return op.vec_size == 1 or (op.mask is not None and X.shape[0] % 2 == 0)


def _is_own(op, colIdx):
    """Is ``colIdx`` the very array that the operator's columns come from (a view of it, as [nnz, 1]), or None?"""
    own = op.colIdx if op.vec_size == 1 else getattr(op, "csr_colIdx", None)
    return own is not None and (colIdx is None or colIdx.dtype == own.dtype and colIdx.numel() == own.numel()
                                and colIdx.data_ptr() == own.data_ptr())


def _slot_columns(op, colIdx):
    """For every score the column the reference's attention-weight gradient multiplies it with (gnn_conv.py:166-172:
    d_attention[mask] times the caller's colIdx in CSR order; 2x1 blocks: zero at padding).  None where that is the entry's own
    column: CSR operators that are given their own array, and the windowed layout, whose entries have an order of their own.  The
    slots of an operator's own columns are made once; other columns are taken as they are at every call."""
    if _fmt(op) == 4:
        return None
    own = _is_own(op, colIdx)
    if op.vec_size == 1:
        return None if own else colIdx.reshape(-1).float()
    k = op.__dict__.get("_own_slot_columns")
    if own and k is not None and k[0] is op.csr_colIdx and k[1] is op.mask:
        return k[2]
    slots = torch.zeros(op.val.numel(), device=op.val.device)
    slots[op.mask] = (op.csr_colIdx if own else colIdx).reshape(-1).float()
    if own:
        op._own_slot_columns = (op.csr_colIdx, op.mask, slots)
    return slots


def _native(op, slots=None):
    """The operator as the extension module's layers take it; made once, and again when anything it is made of changes."""
    arrays = (_row_ptr(op), op.colIdx, op.val, op.target_row if op.if_split else None)
    numbers = (_fmt(op), op.CF, _bw(op), getattr(op, "fold_dense", True))
    k = op.__dict__.get("_native_operator")
    if k is None or k[1] != numbers or k[2] is not slots or any(a is not b for a, b in zip(k[0], arrays)):
        native = SpCONV.Operator(numbers[0], *arrays, *numbers[1:], slots)
        k = op._native_operator = (arrays, numbers, slots, native)
    return k[-1]


class _Recorded(torch.autograd.Function):
    """A native layer or loss as one operation of a trace.  torch.jit.trace records Python functions and ATen operators; of what a
    native node launches it would record the allocations alone."""

    @staticmethod
    def forward(ctx, native, front, *inputs):
        with torch.enable_grad():
            ctx.inputs = [t.detach().requires_grad_(t.requires_grad) if isinstance(t, torch.Tensor) else t for t in inputs]
            ctx.out = native(*front, *ctx.inputs)
        return ctx.out.detach()

    @staticmethod
    def backward(ctx, grad):
        at = [i for i, t in enumerate(ctx.inputs) if isinstance(t, torch.Tensor) and t.requires_grad]
        grads = torch.autograd.grad(ctx.out, [ctx.inputs[i] for i in at], grad, retain_graph=True)
        return (None, None) + tuple(grads[at.index(i)] if i in at else None for i in range(len(ctx.inputs)))


def _run(native, front, *inputs):
    """``native(*front, *inputs)``; ``front``: what comes before the tensors"""
    return _Recorded.apply(native, front, *inputs) if torch.jit.is_tracing() else native(*front, *inputs)


def nll_loss_mean(logp, labels):
    """``F.nll_loss(logp, labels)`` (mean over the rows, the loss of the reference's training step, GNN.py:131-146)
    through the library's kernels.  PyTorch reduces the whole batch in one workgroup -- 1.7 ms per step forward plus
    backward on 10^6 nodes -- where these kernels take some tens of microseconds.  Rows whose label is outside
    [0, C) do not count, as with PyTorch's ignore_index.  Anything but contiguous float32 CUDA log-probabilities with
    int64 labels goes to PyTorch."""
    if (logp.is_cuda and logp.dtype == torch.float32 and logp.dim() == 2 and labels.dtype == torch.int64
            and labels.dim() == 1):
        return _run(SpCONV.nll_loss_layer, (), logp.contiguous(), labels.contiguous())
    return torch.nn.functional.nll_loss(logp, labels)


def softmax_nll_loss_mean(logits, labels):
    """``F.nll_loss(F.log_softmax(logits, dim=1), labels)`` -- the end of the reference's networks and the loss of its
    training step (GNN.py:61,78,101 and 131-146) -- as one function of the logits: one pass over the [n, C] matrix
    forward, one read and one write backward, where the two separate operators make five.  Class counts other than a
    multiple of 4 up to 64, and anything but contiguous float32 CUDA logits with int64 labels, take the separate
    operators."""
    if (logits.is_cuda and logits.dtype == torch.float32 and logits.dim() == 2 and labels.dtype == torch.int64
            and labels.dim() == 1 and SpCONV.softmax_nll_supported(int(logits.shape[1]))):
        return _run(SpCONV.softmax_nll_layer, (), logits.contiguous(), labels.contiguous())
    return nll_loss_mean(torch.nn.functional.log_softmax(logits, dim=1), labels)


class GCNFunction(object):
    """forward A(HW); backward dH = (A dY) W^T, dW = H^T (A dY) -- A is symmetric (gnn_conv.py:13-107)."""

    @staticmethod
    def apply(H, weight, ParamSpMM):
        return _run(SpCONV.gcn_layer, (_native(ParamSpMM),), H, weight)


class GCNAggregateFirstFunction(object):
    """The same layer computed as (A H) W: for a layer that widens its input (in_features < out_features) the sparse
    product then runs at the input's width.  Backward: dW = (A H)^T dY (A H is kept from the forward pass, so the
    weight gradient needs no sparse product) and dH = A (dY W^T), again at the input's width -- A is symmetric, as in
    the reference's own backward (gnn_conv.py:56-107).  ``ParamSpMM`` is the operator configured for the *input*
    width."""

    @staticmethod
    def apply(H, weight, ParamSpMM):
        return _run(SpCONV.gcn_aggregate_first_layer, (_native(ParamSpMM),), H, weight)


class GCNReLUInputFunction(object):
    """The GCN layer reading its input through a ReLU, A (relu(Z) W), as one function of the pre-activation values
    Z: forward relu(Z) W with the activation applied as Z is read; backward dZ = ((A dY) W^T) where Z > 0 and
    dW = relu(Z)^T (A dY), again without a pass for the activation.  Five layers with F.relu between them
    (GNN.py:43-61) are conv1(x), then four of these.  On a windowed operator a square layer of 16 or 32 columns runs
    the dense product inside the sparse kernel."""

    @staticmethod
    def apply(Z, weight, ParamSpMM):
        return _run(SpCONV.gcn_relu_layer, (_native(ParamSpMM),), Z, weight)


class _Layer(torch.nn.Module):
    def __init__(self, input_dim, output_dim):
        super().__init__()
        self.weights = torch.nn.Parameter(torch.randn(input_dim, output_dim))
        self.reset_parameters()

    def reset_parameters(self):
        bound = 1.0 / math.sqrt(self.weights.size(1))
        self.weights.data.uniform_(-bound, bound)

    def _operator(self, spmm_dict):
        width = self.weights.size(1)
        if width not in spmm_dict:
            raise ValueError("SpMMDecider not support dim: " + str(width))
        return spmm_dict[width]


class GCNConv(_Layer):
    aggregate_first = True  # (A H) W where that is the cheaper order and spmm_dict holds an operator for H's width

    def forward(self, H, spmm_dict, relu_input=False):
        """``relu_input``: H holds pre-activation values and the layer computes A (relu(H) W); the activation and its
        backward are folded into the dense products around the sparse one.

        A layer that widens its input is computed as (A H) W when ``spmm_dict`` also holds an operator for the input's
        width (the reference's layers look up the output's width only, gnn_conv.py:121-124, and always compute
        A (H W))."""
        fn, op = self.choose(H.shape[0], spmm_dict, relu_input)
        return fn.apply(H, self.weights, op)

    def choose(self, rows, spmm_dict, relu_input):
        """(function, operator) of a forward pass over ``rows`` rows"""
        in_w, out_w = self.weights.shape
        if self.aggregate_first and not relu_input and in_w < out_w and in_w in spmm_dict:
            return GCNAggregateFirstFunction, spmm_dict[in_w]
        return GCNReLUInputFunction if relu_input else GCNFunction, self._operator(spmm_dict)


class AGNNFunction(object):
    """X' = XW; e = <X'_i, X'_j> per stored entry; attention = e * w; out = SpMM(attention, X')
    (gnn_conv.py:128-180).  No softmax, as in the reference.  ``relu_input``: X holds pre-activation values; the
    activation and its backward ride on the dense products."""

    @staticmethod
    def apply(X, weights, attention_w, ParamSpMM, colIdx, relu_input=False):
        if _attn_fused(ParamSpMM, X, weights):
            # scores (the head's weight multiplied in) and their aggregation in one launch per direction
            native = _native(ParamSpMM, _slot_columns(ParamSpMM, colIdx))
            return _run(SpCONV.agnn_layer, (native,), X, weights, attention_w, bool(relu_input))
        return _AGNNUnfused.apply(X, weights, attention_w, ParamSpMM, colIdx, relu_input)


class _AGNNUnfused(torch.autograd.Function):
    """The layer with its SDDMM and SpMM as separate operators: widths past the fused kernels', double precision."""

    @staticmethod
    def forward(ctx, X, weights, attention_w, ParamSpMM, colIdx, relu_input=False):
        ctx.relu_input = bool(relu_input)
        X_prime = SpCONV.dense_relu_xw(X, weights) if relu_input else SpCONV.dense_xw(X, weights, False)
        if _fmt(ParamSpMM) == 4:
            edge_attentions = ParamSpMM.AGNN_sddmm(X_prime, attention_w.detach().reshape(-1)[:1])
        else:
            edge_feature = ParamSpMM.AGNN_sddmm(X_prime)
            # csr: [nnz] ; 2x1 blocks: [nblk, 2] -- a single head scales both the same way
            edge_attentions = (edge_feature * attention_w.reshape(())).contiguous()
        out = ParamSpMM.AGNN_spmm(edge_attentions, X_prime)
        ctx.save_for_backward(X, weights, edge_attentions)
        ctx.colIdx = colIdx
        ctx.ParamSpMM = ParamSpMM
        return out

    @staticmethod
    def backward(ctx, d_output):
        op = ctx.ParamSpMM
        X, weights, edge_attentions = ctx.saved_tensors
        d_output = d_output.contiguous()
        d_input_prime = op.AGNN_spmm(edge_attentions, d_output)
        if not ctx.needs_input_grad[0]:
            d_input = None
        elif ctx.relu_input:
            d_input = SpCONV.dense_xwt_masked(d_input_prime, weights, X)
        else:
            d_input = SpCONV.dense_xw(d_input_prime, weights, True)
        # X^T * d_input_prime (relu(X)^T when the layer reads X through the activation)
        d_weights = SpCONV.weight_gradient_relu(X, d_input_prime) if ctx.relu_input else SpCONV.weight_gradient(X, d_input_prime)
        d_attention = op.AGNN_sddmm(d_output)
        if d_attention.dim() != 1:
            d_attention = d_attention.view(-1)[op.mask]  # block layout -> CSR slots
        # the reference's literal formula for the attention weight gradient (gnn_conv.py:172):
        # mm(d_attention[1, nnz] expanded to n_heads rows, colIdx.float()[nnz, 1])^T.  Every row of the product is the
        # same dot product over the nnz entries; as a GEMM it takes 20 ms on 2*10^7 entries (a 1 x nnz x 1 problem),
        # as a dot product some tens of microseconds.  A windowed operator keeps its entries in its own order inside the rows:
        # its colIdx is the one that matches.  The float copy of an operator's own columns is made once.
        col = op.colIdx if _fmt(op) == 4 or ctx.colIdx is None else ctx.colIdx
        k = op.__dict__.get("_own_columns_as_float")
        if k is not None and k[0] is op.colIdx and k[1].dtype == d_attention.dtype and k[1].numel() == col.numel() and _is_own(op, col):
            col_f = k[1]
        else:
            col_f = col.reshape(-1).to(d_attention.dtype)
            if _is_own(op, col):
                op._own_columns_as_float = (op.colIdx, col_f)
        d_attention_w = torch.dot(d_attention, col_f).reshape(1, 1).expand(1, n_heads)
        return d_input, d_weights, d_attention_w, None, None, None


class AGNNConv(_Layer):
    def __init__(self, input_dim, output_dim):
        super().__init__(input_dim, output_dim)
        self.attention_w = torch.nn.Parameter(torch.randn(1, n_heads))

    def forward(self, X, spmm_dict, colIdx, relu_input=False):
        return AGNNFunction.apply(X, self.weights, self.attention_w, self._operator(spmm_dict), colIdx, relu_input)


class GINFunction(object):
    """forward (A X) W; backward dW = (A X)^T dY, dX = A (dY W^T) (gnn_conv.py:202-220)."""

    @staticmethod
    def apply(X, weight, ParamSpMM):
        if ParamSpMM.vec_size == 1 or (ParamSpMM.vec_size == 2 and X.shape[0] % 2 == 0):
            return _run(SpCONV.gin_layer, (_native(ParamSpMM),), X, weight)
        return _GINOnOperator.apply(X, weight, ParamSpMM)


class _GINOnOperator(torch.autograd.Function):
    """The same through the operator's own method: 3x1 blocks, and inputs that end inside a block."""

    @staticmethod
    def forward(ctx, X, weight, ParamSpMM):
        X_agg = ParamSpMM.GIN_spmm(X)
        ctx.save_for_backward(X_agg, weight)
        ctx.ParamSpMM = ParamSpMM
        return SpCONV.dense_xw(X_agg, weight, False)

    @staticmethod
    def backward(ctx, d_output):
        X_agg, weights = ctx.saved_tensors
        d_output = d_output.contiguous()  # an upstream gradient may be a view (expand, transpose, slice)
        d_weights = SpCONV.weight_gradient(X_agg, d_output)  # X_agg^T * d_output
        # the network's first layer reads the features, which need no gradient: no dense and no sparse product for it
        d_input = ctx.ParamSpMM.GIN_spmm(SpCONV.dense_xw(d_output, weights, True)) if ctx.needs_input_grad[0] else None
        return d_input, d_weights, None


class GINReLUInputFunction(object):
    """(A relu(Z)) W as one function of the pre-activation values Z, for a layer that widens its input: the activation
    is applied as the sparse product gathers the rows of Z (ParamSpCONV.aggregate_act), the gradient is masked in a pass
    that follows the backward product.  The reference's driver applies F.relu between the layers (GNN.py:63-78)."""

    @staticmethod
    def apply(Z, weight, ParamSpMM):
        return _run(SpCONV.gin_relu_layer, (_native(ParamSpMM),), Z, weight)


class GINConv(_Layer):
    operator_of_input_width = True

    def forward(self, X, spmm_dict, relu_input=False):
        """``relu_input``: X holds pre-activation values and the layer computes (A relu(X)) W without an activation
        pass.  A layer that does not widen its input is evaluated as A (relu(X) W) -- the same product, the sparse
        part at the narrower width -- with the activation and its backward folded into the dense products, like the
        GCN layer; a widening layer applies the activation inside the sparse product."""
        fn, op = self.choose(X.shape[0], spmm_dict, relu_input)
        if relu_input and fn in (GINFunction, _GINOnOperator):
            X = torch.relu(X)
        return fn.apply(X, self.weights, op)

    def choose(self, rows, spmm_dict, relu_input):
        """(function, operator) of a forward pass over ``rows`` rows; functions without ReLU in their name take an
        activated input"""
        in_w, out_w = self.weights.shape
        if relu_input and in_w >= out_w:
            op = self._operator(spmm_dict)
            if op.vec_size in (1, 2):
                return GCNReLUInputFunction, op
        # the sparse product runs at the input's width: take the operator configured for that width when there is
        # one (the reference's layers look up the output's width only, gnn_conv.py:223-226)
        op = spmm_dict[in_w] if self.operator_of_input_width and in_w in spmm_dict else self._operator(spmm_dict)
        if relu_input and op.vec_size in (1, 2):
            return GINReLUInputFunction, op
        return GINFunction if op.vec_size == 1 or (op.vec_size == 2 and rows % 2 == 0) else _GINOnOperator, op


# kinds of ParamSpCONV.network_loss
_NETWORK_KIND = {GCNFunction: 0, GCNAggregateFirstFunction: 1, GINFunction: 1, GCNReLUInputFunction: 2, GINReLUInputFunction: 3}


def network_loss(convs, spmm_dict, x, labels):
    """Layers ``convs`` with ReLU between them on ``x``, log-softmax and mean NLL loss as one autograd node, or None where
    some part of it has to run by itself: subclasses, layers with hooks and weights with hooks (one node hands its gradients out
    together, when the last is formed), operators a layer's native form does not take, losses softmax_nll_loss_mean leaves to
    PyTorch."""
    if torch.jit.is_tracing():
        return None
    if not (x.is_cuda and x.dtype == torch.float32 and x.dim() == 2 and labels.is_cuda and labels.dtype == torch.int64
            and labels.dim() == 1 and labels.is_contiguous() and not _module._has_any_global_hook()):
        return None
    kinds, ops, weights = [], [], []
    for conv in convs:
        w = conv.weights
        if (type(conv) not in (GCNConv, GINConv) or conv._forward_hooks or conv._forward_pre_hooks or conv._backward_hooks
                or conv._backward_pre_hooks or "forward" in conv.__dict__ or w.dtype != torch.float32
                or w._backward_hooks or getattr(w, "_post_accumulate_grad_hooks", None)):
            return None
        fn, op = conv.choose(x.shape[0], spmm_dict, bool(kinds))
        kind = _NETWORK_KIND.get(fn)
        if kind is None or (kinds and kind < 2):
            return None
        kinds.append(kind)
        ops.append(_native(op))
        weights.append(w)
    if not SpCONV.softmax_nll_supported(w.shape[1]):
        return None
    return SpCONV.network_loss(kinds, ops, x, weights, labels)
