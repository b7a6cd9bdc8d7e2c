"""Layer-level operators: autograd functions over the C ABI of libdifflut_hip.so.

These are the callers of the drop-in boundary.  Those that a training step or an inference request is made of are native
(csrc/host_ops.cpp; the classes here give them the call conventions of a torch.autograd.Function), the others are
torch.autograd.Functions over ctypes.  All keep the conventions of the
reference's autograd wrappers (difflut/layers/random_layer.py:34-100,
difflut/nodes/dwn_node.py:58-128, difflut/nodes/probabilistic_node.py:39-129,
difflut/layers/learnable_layer.py:58-123): inputs are made contiguous fp32, outputs
are new tensors, non-tensor arguments get no gradient.  Unlike the reference, one
call covers a whole layer, kernels go to torch's current stream and nothing
synchronises the device.
"""
import torch

from . import _native as nat
from . import cpu_ops

FAST_K = 6


def _f32(t):
    return t if t.dtype is torch.float32 and t.is_contiguous() else t.contiguous().float()


def _bytes(n, device):
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device=device)


def _per_node(values, N, device):
    """A number or tensor of per-node values as the float32 device array [N] the kernels read; what a layer's bank hands
    over is that already (five torch calls less per array)."""
    if (torch.is_tensor(values) and values.dtype is torch.float32 and values.dim() == 1 and values.shape[0] == N
            and values.device == device and not values.requires_grad and values.is_contiguous()):
        return values
    values = torch.as_tensor(values, dtype=torch.float32, device=device).detach()
    return values.reshape(-1).expand(N).contiguous()


class MappingPlan:
    """Device-side form of an index table idx [N,k] over I inputs.

    idx32   int32 [N,k]         the table widened (the reference registers int16 below 32768 inputs)
    inv_ptr int32 [I+1]         CSR row pointers of the inverse mapping
    inv_pos int32 [N*k]         flat positions n*k+j, grouped by input, ascending inside a group
    Built once per table with torch ops (sort + bincount); the kernels only read it.
    """

    ordered = False  # position p reads input p: known of a plan made by in_order()

    def __init__(self, idx, input_size):
        if idx.dim() != 2:
            raise ValueError(f"mapping indices must be 2D (nodes, inputs per node), got {tuple(idx.shape)}")
        if idx.dtype not in (torch.int16, torch.int32, torch.int64):
            raise TypeError(f"mapping indices must be int16, int32 or int64, got {idx.dtype}")
        self.N, self.k = idx.shape
        self.I = int(input_size)
        flat = idx.reshape(-1).long()
        if flat.numel() and (int(flat.min()) < 0 or int(flat.max()) >= self.I):
            raise IndexError(f"mapping index outside [0, {self.I})")
        self.idx32 = idx.to(torch.int32).contiguous()
        order = torch.argsort(flat, stable=True)
        counts = torch.bincount(flat, minlength=self.I)
        self.inv_ptr = torch.cat([counts.new_zeros(1), counts.cumsum(0)]).to(torch.int32).contiguous()
        self.inv_pos = order.to(torch.int32).contiguous()
        self.device = idx.device
        self.source_ptr = idx.data_ptr()
        self.source_version = idx._version

    @property
    def host(self):
        """As the native operators take it."""
        return self.idx32, self.inv_ptr, self.inv_pos, self.I

    def matches(self, idx):
        return (idx.device == self.device and idx.data_ptr() == self.source_ptr
                and idx._version == self.source_version and tuple(idx.shape) == (self.N, self.k))

    @classmethod
    def in_order(cls, N, k, device):
        """The plan of N nodes that take the N*k inputs in order: every one of its tables counts up."""
        plan = cls.__new__(cls)
        plan.N, plan.k, plan.I, plan.device, plan.ordered = N, k, N * k, device, True
        counting = torch.arange(N * k + 1, dtype=torch.int32, device=device)
        plan.inv_ptr, plan.inv_pos = counting, counting[:-1]
        plan.idx32 = plan.inv_pos.view(N, k)
        plan.source_ptr, plan.source_version = plan.idx32.data_ptr(), plan.idx32._version
        return plan

    @staticmethod
    def identity(k, device):
        return MappingPlan(torch.arange(k, dtype=torch.int32, device=device).view(1, k), k)


# ----------------------------------------------------------------------------- gather
class GatherFunction(torch.autograd.Function):
    """m[b,n,j] = x[b, idx[n,j]]  (RandomLayer.get_mapping)."""

    @staticmethod
    def forward(ctx, x, idx, plan):
        nat.require_device(x, idx)
        x = _f32(x)
        B, I = x.shape
        N, k = idx.shape
        bits = {torch.int16: 16, torch.int32: 32}.get(idx.dtype)
        if bits is None:
            raise TypeError("Unsupported index type for mapping kernel. Use int16 or int32.")
        m = torch.empty((B, N, k), dtype=torch.float32, device=x.device)
        nat.check(nat.lib().dl_gather_fwd(nat.ptr(x), nat.ptr(idx.contiguous()), bits, nat.ptr(m), B, I, N, k,
                                          nat.stream()))
        ctx.plan = plan
        ctx.shape = (B, I, N, k)
        return m

    @staticmethod
    def backward(ctx, gm):
        B, I, N, k = ctx.shape
        gm = _f32(gm)
        gx = torch.empty((B, I), dtype=torch.float32, device=gm.device)
        p = ctx.plan
        nat.check(nat.lib().dl_gather_bwd(nat.ptr(gm), nat.ptr(p.inv_ptr), nat.ptr(p.inv_pos), nat.ptr(gx), B, I, N, k,
                                          nat.stream()))
        return gx, None, None


# ----------------------------------------------------------------------------- patches of the convolutional layer
def _flip_bytes(flip, shape):
    """A flip mask as the contiguous byte matrix the kernels read (None stays None)."""
    if flip is None:
        return None
    if tuple(flip.shape) != tuple(shape):
        raise RuntimeError(f"flip mask {tuple(flip.shape)} does not match the patch matrix {tuple(shape)}")
    flip = flip.contiguous()
    return flip.view(torch.uint8) if flip.dtype == torch.bool else flip.to(torch.uint8)


class UnfoldFunction(torch.autograd.Function):
    """x [B,C,H,W] -> patches [B*OH*OW, C*KH*KW] (nn.Unfold, transposed and flattened as
    difflut/layers/convolutional.py:199-205 does); backward folds the patch gradients back.
    `geom` = (KH, KW, SH, SW, PH, PW).  `flip` (optional bool/uint8 [rows, C*KH*KW]): entries of the patch matrix that
    the bit-flip augmentation turns into 1 - value; noise, so the backward ignores it."""

    @staticmethod
    def forward(ctx, x, geom, flip=None):
        nat.require_device(x, flip)
        x = _f32(x)
        B, C, H, W = x.shape
        lib = nat.lib()
        rows = lib.dl_unfold_rows(B, H, W, *geom)
        if rows <= 0:
            raise RuntimeError(f"receptive field {geom[:2]} with stride {geom[2:4]}, padding {geom[4:]} does not fit a "
                               f"{H}x{W} image")
        patches = torch.empty((rows, C * geom[0] * geom[1]), dtype=torch.float32, device=x.device)
        flip = _flip_bytes(flip, patches.shape)
        nat.check(lib.dl_unfold_flip(nat.ptr(x), nat.ptr(flip), nat.ptr(patches), None, B, C, H, W, *geom, nat.stream()))
        ctx.shape, ctx.geom = (B, C, H, W), geom
        return patches

    @staticmethod
    def backward(ctx, gp):
        gp = _f32(gp)
        gx = torch.empty(ctx.shape, dtype=torch.float32, device=gp.device)
        nat.check(nat.lib().dl_fold(nat.ptr(gp), 0, nat.ptr(gx), *ctx.shape, *ctx.geom, nat.stream()))
        return gx, None, None


# ----------------------------------------------------------------------------- DWN
class DWNLayerFunction:
    """y[b, n*O+d] = luts[n,d,addr(b,n)] with the extended-finite-difference backward."""

    @staticmethod
    def apply(x, luts, plan, alpha, beta, beta_abs_max=None):
        """alpha, beta: Python floats for the whole layer, or device tensors [N] with every node's own values
        (then beta_abs_max = max |beta|, a host value)."""
        nat.require_device(x, luts)
        if isinstance(alpha, torch.Tensor) or isinstance(beta, torch.Tensor):
            if any(isinstance(v, torch.Tensor) and v.dim() > 1 for v in (alpha, beta)):
                raise RuntimeError("alpha and beta of a layer are numbers or tensors [N]")
            # (what a layer's bank hands over goes on as it is: the native side looks at it as _per_node would)
            if beta_abs_max is None or not (isinstance(alpha, torch.Tensor) and isinstance(beta, torch.Tensor)):
                alpha, beta = _per_node(alpha, plan.N, x.device), _per_node(beta, plan.N, x.device)
                beta_abs_max = float(beta.abs().max()) if beta_abs_max is None else beta_abs_max
            return nat.host().dwn_layer(x, luts, plan.host, alpha, beta, 0.0, beta_abs_max)
        return nat.host().dwn_layer(x, luts, plan.host, None, None, alpha, beta)


class DWNStackFunction:
    """A chain of RandomLayer + DWN layers in one autograd node.  A following DWN layer only thresholds
    what it is given, so between layers the activations stay bit-planes and the gradients stay
    tile-major: no [B, N] fp32 tensor is written or read except the last layer's output (and the
    first layer's input gradient, if asked for).  Same arithmetic as calling the layers one by one."""

    @staticmethod
    def apply(x, source, plans, scalars, head, *luts):
        """`scalars`: per layer (alpha, beta) as numbers, or (alpha [N], beta [N], max |beta|) with every node's own.
        `head`: None, or (groups, tau) of a GroupSum that follows the last layer: the function then returns
        the [B, groups] sums and neither the last layer's [B, N] output nor its gradient is ever written.
        `source` says what the first layer reads:
        None                  x [B, I] itself;
        a tensor [F, nbits]   thermometer thresholds: x is raw data [B, F], its code is produced directly
                              as bit-planes and x gets no gradient (the code is a step function of it);
        a tuple (KH, KW, SH, SW, PH, PW[, flip])   x is an image batch [B, C, H, W]: the first layer reads its patch
                              matrix (rows = output positions), again produced directly as bit-planes; the
                              input gradient is folded back from the tile-major patch gradient.  `flip`
                              (bool [rows, C*KH*KW], optional): patch entries the bit-flip augmentation inverts."""
        nat.require_device(x, source if torch.is_tensor(source) else None, *luts)
        groups, tau = head if head is not None else (0, 1.0)
        def node_values(v, plan):  # a number stands for every node's value
            return v if torch.is_tensor(v) else _per_node(v, plan.N, x.device)

        values = [(node_values(alpha, p), node_values(beta[0], p), 0.0, beta[1]) if beta[1:] else (None, None, alpha, beta[0])
                  for p, (alpha, *beta) in zip(plans, scalars)]
        thresholds, geom, flip = None, (), None
        if torch.is_tensor(source):
            thresholds = source
        elif source is not None:
            geom, flip = source[:6], source[6] if len(source) > 6 else None
        return nat.host().dwn_stack(x, luts, [p.host for p in plans], values, thresholds, geom, flip, groups, tau)


def dwn_stack_eval(x, thresholds, plans, luts, head=None):
    """Inference through a chain of RandomLayer + DWN layers whose first input is binary: `thresholds` [F, nbits]
    (x is raw data, its thermometer code feeds the first layer) or None (x [B, I] holds exact 0/1 values).
    Activations stay bit-planes between the layers; returns the last layer's 0/1 output [B, N], or with
    `head` = (groups, tau) its GroupSum [B, groups].  Equals calling the layers' eval forward one by one."""
    nat.require_device(x, thresholds, *luts)
    groups, tau = head if head is not None else (0, 1.0)
    return nat.host().dwn_stack_eval(x, thresholds, luts, [p.host for p in plans], groups, tau)


def dwn_layer_eval(x, luts, plan):
    if not x.is_cuda:
        return cpu_ops.dwn_layer_eval(x, luts, plan)
    nat.require_device(x, luts)
    x, luts = _f32(x), _f32(luts)
    B, I = x.shape
    N, O, _ = luts.shape
    y = torch.empty((B, N * O), dtype=torch.float32, device=x.device)
    lib = nat.lib()
    dims = (B, I, N, plan.k, O)
    ws = _bytes(lib.dl_dwn_eval_workspace_bytes(*dims), x.device)
    nat.check(lib.dl_dwn_layer_eval_ws(nat.ptr(x), nat.ptr(plan.idx32), nat.ptr(luts), nat.ptr(y), nat.ptr(ws), ws.numel(),
                                       *dims, nat.stream()))
    return y


# ----------------------------------------------------------------------------- DWN-stable and hybrid nodes
class TableSigmoidFunction:
    """luts = sigmoid(raw_luts), elementwise, for a whole bank of tables at once
    (`_get_luts`, dwn_stable_node.py:289-295, hybrid_node.py:309-315)."""

    @staticmethod
    def apply(raw):
        nat.require_device(raw)
        return nat.host().table_sigmoid(raw)


class DWNStableLayerFunction:
    """Thresholded lookup with the gradient-stabilised backward: the EFD sum weighted 1/(h+1) and
    multiplied, like the table gradient, by the node's gradient scale (dwn_stable_node.py:36-206).
    `scale` is a device tensor [N] (one value per node); it gets no gradient, as in the reference."""

    @staticmethod
    def apply(x, luts, scale, plan):
        nat.require_device(x, luts, scale)
        return nat.host().dwn_stable_layer(x, luts, scale, plan.host)


class HybridLayerFunction:
    """Thresholded lookup forward, probabilistic backward on the real-valued inputs (hybrid_node.py:33-204).  Where a
    backward will follow (`keep_tiles`), the forward re-tiles x for it in the pass that thresholds it."""

    @staticmethod
    def apply(x, luts, plan, keep_tiles=True):
        nat.require_device(x, luts)
        return nat.host().hybrid_layer(x, luts, plan.host, keep_tiles)


# ----------------------------------------------------------------------------- Probabilistic
def _node_temperatures(temperature, N, device):
    """None for one temperature (a number), else the nodes' own values as a float32 device array [N]."""
    if not torch.is_tensor(temperature):
        return None
    return _per_node(temperature, N, device)


class ProbLayerFunction:
    """y[b, n*O+d] = sum_a sigmoid(raw[n,a,d]/T) prod_j (x_j a_j + (1-x_j)(1-a_j)); `temperature` is a number for the
    whole layer or a tensor [N] with every node's own value."""

    @staticmethod
    def apply(x, raw, plan, temperature):
        nat.require_device(x, raw)
        if isinstance(temperature, torch.Tensor):
            return nat.host().prob_layer(x, raw, plan.host, plan.ordered, temperature, 0.0)
        return nat.host().prob_layer(x, raw, plan.host, plan.ordered, None, temperature)


def prob_layer_eval(x, raw, plan, temperature):
    if not x.is_cuda:
        return cpu_ops.prob_layer_eval(x, raw, plan, temperature)
    nat.require_device(x, raw)
    x, raw = _f32(x), _f32(raw)
    B, I = x.shape
    N, _, O = raw.shape
    y = torch.empty((B, N * O), dtype=torch.float32, device=x.device)
    lib = nat.lib()
    dims = (B, I, N, plan.k, O)
    ws = _bytes(lib.dl_prob_eval_workspace_bytes(*dims), x.device)
    T = _node_temperatures(temperature, N, x.device)
    if T is None:
        nat.check(lib.dl_prob_layer_eval_ws(nat.ptr(x), nat.ptr(plan.idx32), nat.ptr(raw), float(temperature), nat.ptr(y),
                                            nat.ptr(ws), ws.numel(), *dims, nat.stream()))
    else:
        nat.check(lib.dl_prob_layer_eval_ws_nodes(nat.ptr(x), nat.ptr(plan.idx32), nat.ptr(raw), nat.ptr(T), nat.ptr(y),
                                                  nat.ptr(ws), ws.numel(), *dims, nat.stream()))
    return y


# ----------------------------------------------------------------------------- Learnable mapping
class SoftMapFunction:
    """m = x @ softmax(W / tau, dim=-1).T.  The softmax numerators are kept as 16-bit planes from forward to backward: 6 bytes per
    entry of W with fp32 operands (precision 0: three bf16 planes, or two fp16 halves in the same room), 2 with bf16."""

    @staticmethod
    def apply(x, W, tau, precision):
        nat.require_device(x, W)
        return nat.host().soft_map(x, W, tau, precision)


def row_argmax(W):
    if not W.is_cuda:
        return cpu_ops.row_argmax(W)
    nat.require_device(W)
    W = _f32(W)
    sel = torch.empty((W.shape[0],), dtype=torch.int32, device=W.device)
    nat.check(nat.lib().dl_row_argmax(nat.ptr(W), nat.ptr(sel), W.shape[0], W.shape[1], nat.stream()))
    return sel


class HardSelectFunction(torch.autograd.Function):
    """m[b,o] = x[b, sel[o]] with the straight scatter-add backward."""

    @staticmethod
    def forward(ctx, x, sel, plan):
        nat.require_device(x, sel)
        x = _f32(x)
        B, I = x.shape
        M = sel.numel()
        m = torch.empty((B, M), dtype=torch.float32, device=x.device)
        nat.check(nat.lib().dl_hard_select_fwd(nat.ptr(x), nat.ptr(sel.contiguous().int()), nat.ptr(m), B, I, M,
                                               nat.stream()))
        ctx.plan, ctx.shape = plan, (B, I, M)
        return m

    @staticmethod
    def backward(ctx, gm):
        B, I, M = ctx.shape
        gm = _f32(gm)
        gx = torch.empty((B, I), dtype=torch.float32, device=gm.device)
        p = ctx.plan
        nat.check(nat.lib().dl_hard_select_bwd(nat.ptr(gm), nat.ptr(p.inv_ptr), nat.ptr(p.inv_pos), nat.ptr(gx), B, I, M,
                                               nat.stream()))
        return gx, None, None


# ----------------------------------------------------------------------------- encoder / head
def thermometer_encode(x, thresholds):
    if not x.is_cuda:
        return cpu_ops.thermometer_encode(x, thresholds)
    nat.require_device(x, thresholds)
    x, thr = _f32(x), _f32(thresholds)
    B, F = x.shape
    nbits = thr.shape[1]
    bits = torch.empty((B, F, nbits), dtype=torch.float32, device=x.device)
    nat.check(nat.lib().dl_thermometer_encode(nat.ptr(x), nat.ptr(thr), nat.ptr(bits), B, F, nbits, nat.stream()))
    return bits


class CrossEntropyFunction:
    """Mean cross-entropy of [B, C] logits against int64 class labels: loss and its gradient from one pass
    (what torch.nn.functional.cross_entropy and its backward compute for the logits GroupSum returns)."""

    @staticmethod
    def apply(logits, labels):
        nat.require_device(logits, labels)
        return nat.host().cross_entropy(logits, labels)


class GroupSumFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, groups, tau):
        nat.require_device(x)
        x = _f32(x)
        B, F = x.shape
        y = torch.empty((B, groups), dtype=torch.float32, device=x.device)
        nat.check(nat.lib().dl_group_sum_fwd(nat.ptr(x), nat.ptr(y), B, F, groups, float(tau), nat.stream()))
        ctx.args = (B, F, groups, float(tau))
        return y

    @staticmethod
    def backward(ctx, gy):
        B, F, groups, tau = ctx.args
        gy = _f32(gy)
        gx = torch.empty((B, F), dtype=torch.float32, device=gy.device)
        nat.check(nat.lib().dl_group_sum_bwd(nat.ptr(gy), nat.ptr(gx), B, F, groups, tau, nat.stream()))
        return gx, None, None


# ----------------------------------------------------------------------------- dispatch
# The reference's rule (random_layer.py:272, dwn_node.py:334, probabilistic_node.py:277): the extension runs iff the
# input is a device tensor, otherwise the CPU code does.  Layers, nodes, the encoder and the head call these.
def gather(x, idx, plan):
    return GatherFunction.apply(x, idx, plan) if x.is_cuda else cpu_ops.gather(x, idx)


def dwn_layer(x, luts, plan, alpha, beta, beta_abs_max=None):
    if x.is_cuda:
        return DWNLayerFunction.apply(x, luts, plan, alpha, beta, beta_abs_max)
    return cpu_ops.dwn_layer(x, luts, plan, alpha, beta)


def dwn_stable_layer(x, luts, scale, plan):
    return DWNStableLayerFunction.apply(x, luts, scale, plan) if x.is_cuda else cpu_ops.dwn_stable_layer(x, luts, scale, plan)


def hybrid_layer(x, luts, plan):
    if not x.is_cuda:
        return cpu_ops.hybrid_layer(x, luts, plan)
    keep = torch.is_grad_enabled() and (x.requires_grad or luts.requires_grad)  # a backward may follow
    return HybridLayerFunction.apply(x, luts, plan, keep)


def dwn_stable_raw_layer(x, raw, scale, plan):
    """dwn_stable_layer(x, table_sigmoid(raw), scale, plan), as one operator."""
    if not x.is_cuda:
        return cpu_ops.dwn_stable_layer(x, table_sigmoid(raw), scale, plan)
    return nat.host().dwn_stable_raw_layer(x, raw, scale, plan.host)


def hybrid_raw_layer(x, raw, plan):
    """hybrid_layer(x, table_sigmoid(raw), plan), as one operator."""
    if not x.is_cuda:
        return cpu_ops.hybrid_layer(x, table_sigmoid(raw), plan)
    keep = torch.is_grad_enabled() and (x.requires_grad or raw.requires_grad)
    return nat.host().hybrid_raw_layer(x, raw, plan.host, keep)


def table_sigmoid(raw):
    return TableSigmoidFunction.apply(raw) if raw.is_cuda else torch.sigmoid(raw.float())


def prob_layer(x, raw, plan, temperature):
    return ProbLayerFunction.apply(x, raw, plan, temperature) if x.is_cuda else cpu_ops.prob_layer(x, raw, plan, temperature)


def soft_map(x, W, tau, precision=0):
    return SoftMapFunction.apply(x, W, tau, precision) if x.is_cuda else cpu_ops.soft_map(x, W, tau, precision)


def hard_select(x, sel, plan):
    return HardSelectFunction.apply(x, sel, plan) if x.is_cuda else cpu_ops.hard_select(x, sel)


def unfold(x, geom, flip=None):
    """Patch matrix [B*OH*OW, C*KH*KW] of an image batch; on the CPU nn.functional.unfold, transposed and flattened
    as convolutional.py:199-205 does, with the flip applied to the patches."""
    if x.is_cuda:
        return UnfoldFunction.apply(x, geom, flip)
    kh, kw, sh, sw, ph, pw = geom
    cols = torch.nn.functional.unfold(x.float(), (kh, kw), padding=(ph, pw), stride=(sh, sw))
    patches = cols.transpose(1, 2).reshape(-1, cols.shape[1])
    if flip is not None:
        patches = patches + torch.where(flip.bool(), 1.0 - 2.0 * patches.detach(), torch.zeros_like(patches))
    return patches


def grad_stabilize(grad, per_row, target_std, subtract_mean, eps):
    """(grad - mean) * sqrt(target_std / (mean((grad - mean)^2) + eps)) for a [rows, cols] gradient on the device, over
    the whole tensor or per row (base_layer.py:266-339); a new tensor."""
    nat.require_device(grad)
    g = _f32(grad)
    rows, cols = g.shape
    out = torch.empty_like(g)
    lib = nat.lib()
    ws = _bytes(lib.dl_grad_stabilize_workspace_bytes(rows, cols, int(per_row)), g.device)
    nat.check(lib.dl_grad_stabilize(nat.ptr(g), nat.ptr(out), rows, cols, int(per_row), float(target_std),
                                    int(bool(subtract_mean)), float(eps), nat.ptr(ws), ws.numel(), nat.stream()))
    return out


def group_sum(x, groups, tau):
    return GroupSumFunction.apply(x, groups, tau) if x.is_cuda else cpu_ops.group_sum(x, groups, tau)


def cross_entropy(logits, labels):
    if logits.is_cuda:
        return CrossEntropyFunction.apply(logits, labels)
    return torch.nn.functional.cross_entropy(logits.float(), labels.long())
