"""Fused q/k/v and gate/up projections: one 4-bit launch instead of three / two, and the whole MLP decode step in one.

Counterpart of make_quant_attn / make_fused_mlp (src/alpaca_lora_4bit/model_attn_mlp_patch.py:73-247 of the
reference), which concatenate the packed tensors of the projections along N and swap in their own attention / MLP
classes.  Two ways here, both leaving the host model's own attention / MLP code in charge:

* in place (the default): the projections stay where they are, on their OWN tensors, and become members of a group.
  At decode sizes (up to 16 rows, no grad) the first member called runs ONE grouped launch for all of them
  (quant_hip.gemv_grouped -> q4_gemv_grouped_f16) and the others pick their result up.  No second copy of the
  weights, the state dict keeps its keys, and members may be LoRA layers (Linear4bitLt): the grouped launch does the
  base products, each member adds its own adapter.  make_fused_mlp also routes the block's forward, at decode sizes,
  through quant_hip.mlp_decode (gate, up, silu(gate) * up and down in one launch) or quant_hip.mlp_rows (two launches).
* `concatenate=True`: the reference's layout.  One new layer holds the N-concatenated tensors and each projection is
  replaced by a slice view of its output (one wider GEMM at prefill sizes as well); `inject_lora_layers(model,
  lora_path)` (model_attn_mlp_patch.py:283-335) then puts a saved q/v adapter onto the fused qkv layer as ONE
  adapter of rank r_q + r_v whose B matrix is block-structured (zero rows for k_proj).
"""
import json
import os
import re
import threading

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import autograd_4bit, matmul_utils_4bit
from .autograd_4bit import Autograd4bitQuantLinear, _buffer, _has_bias, _weight, fuse_quant_linears


def _where(x):
    """The thread, the stream and whether it is being captured: what is queued here is there for callers of the same only."""
    if not x.is_cuda:
        return threading.get_ident(), 0, False
    return threading.get_ident(), torch._C._cuda_getCurrentRawStream(x.get_device()), torch.cuda.is_current_stream_capturing()


class _Held:
    """Outputs for one input that members of a group have not called for yet, put in place by one assignment."""
    __slots__ = ('x', 'key', 'where', 'outs', 'adapted', 'left', 'layers', 'invalidations')

    def __init__(self, x, key, outs, left, layers=None):
        self.x, self.key, self.where = x, key, _where(x)
        self.outs, self.adapted, self.left = outs, [None] * len(outs), left
        self.layers, self.invalidations = layers, matmul_utils_4bit.quant_hip.invalidations


class FusedProjectionSlice(nn.Module):
    """Stands where one projection of a fused group stood; returns its columns of the fused output.
    The fused layer itself is registered once, on the parent module; the slices only point to it."""

    def __init__(self, group, start, stop):
        super().__init__()
        object.__setattr__(self, "_group", group)          # not a registered submodule: no duplicate state
        self.in_features = group.layer.in_features
        self.out_features = stop - start
        self._start, self._stop = start, stop

    def forward(self, x):
        y = self._group.run(x)
        return y[..., self._start:self._stop]


class _FusedGroup:
    """Runs the fused layer once per input tensor and hands the result to every slice.  The result is kept for as
    long as the same tensor object comes back unmodified in the same grad mode (identity, in-place version counter),
    whatever the order in which the host block calls its projections, and dropped as soon as every slice has been
    served or the block returns (forward hook installed by _fuse_children), so nothing stays pinned between forwards.
    Another thread, stream or capture than the one that ran the layer runs it again."""

    def __init__(self, layer, n_slices):
        self.layer = layer
        self.n_slices = n_slices
        self.hook = None
        self.clear()

    def run(self, x):
        if x.is_inference():
            return self.layer(x)                             # no version counter to hold a result by
        h = self._now
        if h is None or h.x is not x or h.key != (x._version, torch.is_grad_enabled()) or h.where != _where(x):
            h = self._now = _Held(x, (x._version, torch.is_grad_enabled()), [self.layer(x)], self.n_slices)
        y = h.outs[0]
        h.left -= 1
        if not h.left and self._now is h:
            self._now = None
        return y

    _x = property(lambda self: None if self._now is None else self._now.x)
    _y = property(lambda self: None if self._now is None else self._now.outs[0])

    def clear(self, *unused):
        self._now = None


_ADAPTER_TYPES = (torch.float16, torch.float32)


def _same_adapter(p, q):
    return p[0] is q[0] and p[1] is q[1] and p[2:] == q[2:]


def _layer_key(m):
    """What is kept about layer `m` rests on: its buffers and their contents as the version counters show them.  Writes that these
    do not show are what quant_hip.invalidate is for; its count is compared beside this."""
    b = m._buffers
    q, z, s, g = b.get('qweight'), b.get('qzeros'), b.get('scales'), b.get('g_idx')
    return q, z, s, g, q._version, z._version, s._version, -1 if g is None else g._version


def _same_layer(m, k):
    """_layer_key(m) is `k`, without building it."""
    b = m._buffers
    q, z, s, g, vq, vz, vs, vg = k
    return (b.get('qweight') is q and b.get('qzeros') is z and b.get('scales') is s and b.get('g_idx') is g and s._version == vs
            and q._version == vq and z._version == vz and (g is None or g._version == vg))


class _MemberGroup:
    """Projections that share their input (q|k|v, gate|up), each on its own tensors.  `run(member, x)` is called from
    Autograd4bitQuantLinear.forward at decode sizes: the first call for an input runs one grouped launch for all
    members, every member takes its own output tensor exactly once (callers add bias and adapter in place; `run_adapted`
    adds the adapters of all members in one more launch)."""

    def __init__(self, members):
        self.members = list(members)
        self.index = {id(m): i for i, m in enumerate(self.members)}
        self.groupsize = self.members[0].groupsize
        self.usable = None                                   # decided at the first call (needs the tensors on the GPU)
        self._layer_cache = self._keys = None
        self._invalidations = -1
        self._gemm_ok = None                                 # sequential groups AND scales below 64 (the tiled kernels' fused form)
        self.hook = None
        self.clear()

    def _check(self):
        from . import quant_hip
        try:
            for m in self.members:
                info = quant_hip._layer_info(m.qweight, m.qzeros, m.scales if m.scales.dtype == torch.float16 else m.scales.half(),
                                             m.g_idx, m.groupsize)
                if info.plan is not None or info.gemv_gidx is not None:
                    return False                             # act-order members keep their own launches
        except Exception:
            return False
        return all(m.scales.dtype == torch.float16 for m in self.members)

    def _layers(self):
        """(qweight, qzeros, scales) of every member, rebuilt when a member's buffers were replaced (a cast, a reload) or written in
        place, or `quant_hip.invalidate` was called."""
        if self._layer_cache is not None and self._invalidations == matmul_utils_4bit.quant_hip.invalidations:
            for m, (q, z, s, g, vq, vz, vs, vg) in zip(self.members, self._keys):
                b = m._buffers                               # _same_layer, without a call per member
                if (b.get('qweight') is not q or b.get('qzeros') is not z or b.get('scales') is not s or b.get('g_idx') is not g
                        or s._version != vs or q._version != vq or z._version != vz or (g is not None and g._version != vg)):
                    break
            else:
                return self._layer_cache
        self.clear()                                         # outputs of the tensors as they were
        self.usable = self._check()
        self._gemm_ok = None
        self._keys = [_layer_key(m) for m in self.members] if self.usable else None
        self._invalidations = matmul_utils_4bit.quant_hip.invalidations
        layers = self._layer_cache = [(m.qweight, m.qzeros, m.scales) for m in self.members] if self.usable else None
        return layers                                        # last, so that another thread finds the keys of what it finds

    def run(self, member, x):
        if x.is_inference():
            return None                                      # writes to x cannot be told from its version: nothing is held for it
        i = self.index[id(member)]
        h = self._held(i, x)
        if h is None or h.adapted[i] is not None:
            layers = self._layers()
            if layers is None:
                return None
            h = self._launch(x, layers)
        return self._take(h, i)

    def _held(self, i, x):
        """Member i's output for x is there, of the tensors that the member has now and for this thread, stream and capture."""
        h = self._now
        if h is not None and h.x is x and h.key == x._version and h.outs[i] is not None and self._same(h, i) and h.where == _where(x):
            return h
        return None

    def _same(self, h, i):
        return h.invalidations == matmul_utils_4bit.quant_hip.invalidations and _same_layer(self.members[i], h.layers[i])

    def _launch(self, x, layers):
        # the compiled binding checks shapes, dtypes and devices; sequential groups were established by _check()
        outs = matmul_utils_4bit.quant_hip.gemv_grouped_prepared(x, layers, self.groupsize)
        if x.dim() != 2:
            lead = tuple(x.shape[:-1])
            outs = [o.view(lead + (o.shape[-1],)) for o in outs]
        h = self._now = _Held(x, x._version, outs, len(outs), self._keys)
        return h

    def _take(self, h, i):
        y, h.outs[i], h.adapted[i] = h.outs[i], None, None
        h.left -= 1
        if not h.left and self._now is h:
            self._now = None
        return y

    def run_adapted(self, member, x, name):
        """`run` for a member whose adapter `name` is to be added (decode sizes): the products of all members in one launch and
        the adapters of all members in the next, each member picks its finished output up.  None when the group does not take
        this call.  An output that was finished with another adapter than the member now asks for is not handed out: other matrices,
        other storage, a write that the version counters show or that quant_hip.invalidate was told of."""
        adapter = None if x.is_inference() else self._adapter(member, name, x)
        if adapter is None:
            return None
        i = self.index[id(member)]
        h = self._held(i, x)
        if h is None or (h.adapted[i] is not None and not _same_adapter(h.adapted[i], adapter)):
            layers = self._layers()
            if layers is None:
                return None
            h = self._launch(x, layers)
        if h.adapted[i] is None:
            todo = {i: adapter}
            for j, m in enumerate(self.members):
                if j != i and h.outs[j] is not None and h.adapted[j] is None and type(m) is type(member) and not m.disable_adapters:
                    other = m._decode_adapter(x)
                    ad = None if other is None else self._adapter(m, other, x)
                    if ad is not None:
                        todo[j] = ad
            try:
                flat = x.dim() == 2
                matmul_utils_4bit.quant_hip.lora_update_grouped(
                    x if flat and x.is_contiguous() else x.reshape(-1, x.shape[-1]).contiguous(),
                    [(ad[0], ad[1], h.outs[j] if flat else h.outs[j].view(-1, h.outs[j].shape[-1]), ad[2]) for j, ad in todo.items()])
            except BaseException:
                self.clear()                                 # some outputs may have been updated
                raise
            for j, ad in todo.items():
                h.adapted[j] = ad
        return self._take(h, i)

    @staticmethod
    def _adapter(m, name, x):
        """(A, B, scaling, what their contents are known by) of member m's adapter as the grouped update takes it, or None."""
        if _has_bias(m):
            return None                                      # the bias comes between the product and the update
        mods = m._modules
        a, b, dev = _weight(mods['lora_A']._modules[name]), _weight(mods['lora_B']._modules[name]), x.get_device()
        for w in (a, b):
            if w.get_device() != dev or w.dtype not in _ADAPTER_TYPES or w.is_inference():
                return None
        return a, b, float(m.scaling[name]), (a._version, b._version, a.data_ptr(), b.data_ptr(), matmul_utils_4bit.quant_hip.invalidations)

    def _gemm_spec(self, m, x):
        """How member `m` enters a grouped GEMM for input x: (bias | None, lora_A | None, lora_B | None, scaling, drop_p)."""
        bias = _buffer(m, 'bias') if _has_bias(m) else None
        name = None
        if type(m) is not Autograd4bitQuantLinear and not getattr(m, 'disable_adapters', False):
            name = m._fusable_adapter(x)                     # the adapter rides in the launch; otherwise the layer adds it
        if name is None:
            return (bias, None, None, None, 0.0)
        return (bias, _weight(m._modules['lora_A']._modules[name]), _weight(m._modules['lora_B']._modules[name]), float(m.scaling[name]), m._dropout_p(name))

    def run_gemm(self, member, x):
        """Above the decode sizes: ONE grouped GEMM launch for all members (under autograd one node, whose backward is
        one grouped grad-input launch).  Returns the member's output, bias and fused adapter included, or None when
        the group does not take this call (the member then runs by itself)."""
        if x.is_inference():
            return None
        i = self.index[id(member)]
        key = (x._version, torch.is_grad_enabled())
        h = self._gemm_now
        if h is not None and h.x is x and h.key == key and h.outs[i] is not None and self._same(h, i) and h.where == _where(x):
            y, h.outs[i] = h.outs[i], None
            h.left -= 1
            if not h.left and self._gemm_now is h:
                self._gemm_now = None
            return y
        from . import quant_hip
        layers = self._layers()
        if layers is None or not x.is_cuda or x.shape[-1] != member.in_features:
            return None
        rows = x.numel() // member.in_features
        if rows <= quant_hip.MAX_GEMV_ROWS or not (x.dtype == torch.float16 or torch.is_autocast_enabled('cuda')):
            return None
        if matmul_utils_4bit.use_dense_route(rows) or member.in_features % 128 or any(m.out_features % 128 for m in self.members):
            return None
        Ns = [m.out_features for m in self.members]
        if not quant_hip.gemm_grouped_applicable(True, rows, member.in_features, Ns):
            return None
        parts = [self._gemm_spec(m, x) for m in self.members]
        train = torch.is_grad_enabled() and (x.requires_grad or any(
            t is not None and t.requires_grad for _, la, lb, _, _ in parts for t in (la, lb)))
        if train:
            if not quant_hip.gemm_grouped_applicable(False, rows, member.in_features, Ns):
                return None
        elif all(la is None for _, la, _, _, _ in parts) and quant_hip.streams_forward(rows, member.in_features, Ns, self.groupsize):
            # nothing to differentiate and no adapter in the launch: layers that all have a whole-reduction streaming
            # kernel run by themselves.  us apart against grouped: q|k|v of 4096 features at 136 / 200 / 256 rows 41.6 / 49.7 /
            # 52.6 against 48.6 / 49.5 / 50.0, of 5120 at 136 rows 52.2 against 59.6.  Where one of them has none, the
            # group wins (5120, 200 rows: 78.8 against 61.0; gate|up of 4096 -> 11008, 200 rows: 71.8 against 53.2), and with
            # adapters always (q|k|v of 4096, 200 rows: 67.9 against 54.9).
            return None
        if self._gemm_ok is None:
            self._gemm_ok = all(quant_hip._group_layer_ok(l, self.groupsize) for l in layers)
        if not self._gemm_ok:
            return None
        specs, tensors = [], []
        for (qweight, qzeros, scales), (bias, la, lb, scaling, drop_p) in zip(layers, parts):
            seed = int(torch.randint(0, 2 ** 62, (1,)).item()) if drop_p > 0.0 else 0
            specs.append((scaling, drop_p, seed))
            tensors += [qweight, scales, qzeros, bias, la, lb]
        outs = autograd_4bit.AutogradMatmul4bitGroup.apply(x, self.groupsize, tuple(specs), *tensors)
        h = _Held(x, key, list(outs), len(outs) - 1, self._keys)
        y, h.outs[i] = h.outs[i], None
        self._gemm_now = h
        return y

    _x = property(lambda self: None if self._now is None else self._now.x)

    def clear(self, *unused):
        self._now = self._gemm_now = None

    def replace(self, old, new):
        """`new` (for instance a LoRA layer sharing `old`'s packed tensors) takes `old`'s place in the group."""
        i = self.index.pop(id(old))
        old.__dict__.pop('_q4_group', None)
        self.members[i] = new
        self.index[id(new)] = i
        new.__dict__['_q4_group'] = self
        self.usable = None
        self._layer_cache = self._keys = None
        self.clear()


def _fusable(mods):
    if not all(type(m) is Autograd4bitQuantLinear for m in mods):
        return False                                         # LoRA-wrapped or dense projections stay as they are
    first = mods[0]
    return all((m.in_features, m.groupsize, m.bits) == (first.in_features, first.groupsize, first.bits)
               and not m.is_v1_model and torch.equal(m.g_idx, first.g_idx) for m in mods)


def _fuse_children(parent, names, fused_name):
    mods = [getattr(parent, n, None) for n in names]
    if any(m is None for m in mods) or not _fusable(mods):
        return False
    fused = fuse_quant_linears(mods)
    group = _FusedGroup(fused, len(names))
    setattr(parent, fused_name, fused)
    group.hook = parent.register_forward_hook(group.clear)
    start = 0
    for i, (n, m) in enumerate(zip(names, mods)):
        setattr(parent, n, FusedProjectionSlice(group, start, start + m.out_features))
        start += m.out_features
    return True


def _groupable(mods):
    if not all(isinstance(m, Autograd4bitQuantLinear) for m in mods):
        return False                                         # dense projections stay as they are
    first = mods[0]
    return all((m.in_features, m.groupsize, m.bits) == (first.in_features, first.groupsize, first.bits)
               and m.bits == 4 and not m.is_v1_model and m.__dict__.get('_q4_group') is None for m in mods)


def _group_children(parent, names):
    """In-place grouping: the projections keep their tensors and their place; returns the group or None."""
    mods = [getattr(parent, n, None) for n in names]
    if any(m is None for m in mods) or not _groupable(mods):
        return None
    group = _MemberGroup(mods)
    for m in mods:
        m.__dict__['_q4_group'] = group                      # a plain attribute: neither a parameter nor a submodule
    group.hook = parent.register_forward_hook(group.clear)
    return group


def ungroup(model):
    """Undo the in-place grouping (and the MLP decode routing) made by make_quant_attn / make_fused_mlp."""
    count = 0
    for m in model.modules():
        group = m.__dict__.pop('_q4_group', None)
        if group is not None and group.hook is not None:
            group.hook.remove()
            group.hook = None
            count += 1
        if '_q4_mlp_forward' in m.__dict__:
            del m.__dict__['_q4_mlp_forward']
            del m.__dict__['forward']
            m.__dict__.pop('_q4_mlp_args', None)
            m.__dict__.pop('_q4_mlp_gated', None)
    return count


def make_quant_attn(model, is_v1_model=False, concatenate=False):
    """One launch for q_proj / k_proj / v_proj of every attention block (model_attn_mlp_patch.py:73-160).
    Returns the number of blocks changed.  In place by default (see the module docstring); `concatenate=True` builds
    the reference's N-concatenated layer and, like the reference (model_attn_mlp_patch.py:78), turns the shared dense
    buffer off -- process-wide: above matmul_utils_4bit.dense_switch_rows rows every product then allocates its own
    dense buffer; set matmul_utils_4bit.cache_buffer = True again if prefill batches of that size matter."""
    if is_v1_model:
        raise NotImplementedError("v1 (fp zeros) layers are not fused")
    names = ("q_proj", "k_proj", "v_proj")
    count = 0
    if concatenate:
        matmul_utils_4bit.cache_buffer = False
    for m in list(model.modules()):
        if all(hasattr(m, n) for n in names):
            count += bool(_fuse_children(m, names, "qkv_proj") if concatenate else _group_children(m, names))
    if concatenate and torch.cuda.is_available():
        torch.cuda.empty_cache()
    return count


# Up to so many rows the MLP step runs on the block's three layers directly, whatever the block's own forward looks like
# (make_fused_mlp's premise); more rows only where that forward is known to compute the same.
mlp_decode_max_rows = 4


class _GatedForward:
    """The forwards of a gated MLP block whose steps may run fused at any number of rows: compared by their code."""

    def returned(self, x):
        return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))

    def assigned(self, x):
        down_proj = self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))
        return down_proj


def _is_gated_forward(forward):
    """True when `forward` (a bound method) is down_proj(act_fn(gate_proj(x)) * up_proj(x)) and nothing else."""
    code = getattr(getattr(forward, '__func__', None), '__code__', None)
    if code is None:
        return False

    return any(_code_key(code) == _code_key(f.__code__) for f in (_GatedForward.returned, _GatedForward.assigned))


def _steps_unobserved(mlp):
    """No hook and no replaced forward on the block's four steps, which a fused step would pass by."""
    mods = mlp._modules
    for name in ('gate_proj', 'up_proj', 'down_proj', 'act_fn'):
        m = mods.get(name)
        if m is None or m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or 'forward' in m.__dict__:
            return False
    return _is_silu(mods['act_fn']) and not torch.nn.modules.module._has_any_global_hook()


def _code_key(c):
    return (c.co_code, c.co_names, c.co_consts[1:], c.co_argcount, c.co_kwonlyargcount, c.co_flags & 0x0F, c.co_freevars)


class _SiluForward:
    """The forwards of activation modules that are silu and nothing else: compared by their code."""

    def functional(self, input):
        return nn.functional.silu(input)

    def short(self, input):
        return F.silu(input)


_SILU, _SILU_MODULE = F.silu, nn.SiLU.forward
_SILU_FUNCTIONAL, _SILU_SHORT = _code_key(_SiluForward.functional.__code__), _code_key(_SiluForward.short.__code__)


def _is_silu(act):
    """True for silu itself and for a module whose class runs exactly that: nn.SiLU and classes with its forward, or with one that is
    `return nn.functional.silu(input)` (transformers' SiLUActivation).  The class's name or base says nothing about its forward."""
    if F.silu is not _SILU:
        return False                                         # somebody replaced it
    if act is _SILU:
        return True
    if not isinstance(act, nn.Module) or 'forward' in act.__dict__ or type(act).__call__ is not nn.Module.__call__:
        return False
    forward = type(act).forward
    if forward is _SILU_MODULE:
        return True
    code = getattr(forward, '__code__', None)
    if code is None:
        return False
    key = _code_key(code)
    return (key == _SILU_FUNCTIONAL and forward.__globals__.get('nn') is nn) or (key == _SILU_SHORT and forward.__globals__.get('F') is F)


def _plain_no_bias(layer):
    """A 4-bit layer whose forward is the bare product: no active adapter, no bias to add."""
    from .autograd_4bit import _is_all_zero
    if type(layer) is not Autograd4bitQuantLinear:
        if not getattr(layer, 'disable_adapters', False):
            return False
    return layer.disable_bias or _is_all_zero(layer.bias)


class _SiluMul(torch.autograd.Function):
    """silu(gate) * up, one pass forward and one backward; keeps gate and up."""

    @staticmethod
    def forward(ctx, gate, up):
        from . import quant_hip
        ctx.save_for_backward(gate, up)
        return quant_hip.silu_mul(gate, up)

    @staticmethod
    def backward(ctx, dout):
        from . import quant_hip
        gate, up = ctx.saved_tensors
        if torch.is_grad_enabled():                          # a graph of the backward is wanted: the operations it replaces
            out = nn.functional.silu(gate) * up
            wanted = [t for t, need in zip((gate, up), ctx.needs_input_grad) if need]
            grads = list(torch.autograd.grad(out, wanted, dout, create_graph=True))
            return tuple(grads.pop(0) if need else None for need in ctx.needs_input_grad)
        dout = dout.contiguous()
        if not quant_hip.silu_mul_takes(dout, gate):
            return torch.ops.aten.silu_backward(dout * up, gate), dout * nn.functional.silu(gate)
        return quant_hip.silu_mul_bwd(dout, gate, up)


def _gated_rows_forward(mlp, x):
    """The block's forward above the decode sizes: its own three layers, silu(gate) * up in one pass (us, forward / backward, 1024 x
    11008: 24 / 37 as five elementwise kernels, 16 / 24 as two).  Only for forwards known to be this expression."""
    from . import quant_hip
    gate, up = mlp.gate_proj(x), mlp.up_proj(x)
    if not quant_hip.silu_mul_takes(gate, up):
        return mlp.down_proj(mlp.act_fn(gate) * up)
    return mlp.down_proj(_SiluMul.apply(gate, up) if torch.is_grad_enabled() else quant_hip.silu_mul(gate, up))


def _act_unobserved(mlp):
    """The block's activation is a SiLU that nothing hooks, and nothing traces the block."""
    act = mlp._modules.get('act_fn')
    return (act is not None and _is_silu(act) and not act._forward_hooks and not act._forward_pre_hooks and not act._backward_hooks
            and not act._backward_pre_hooks and 'forward' not in act.__dict__ and not torch.nn.modules.module._has_any_global_hook()
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def _mlp_decode_args(mlp):
    """(gate, up, down, groupsize, H) for quant_hip's one-launch MLP step, or None when the block does not qualify right
    now: all three layers plain 4-bit products (no active adapter, no bias to add), fp16 scales, sequential groups."""
    from . import quant_hip
    gate, up, down = mlp.gate_proj, mlp.up_proj, mlp.down_proj
    group = gate.__dict__.get('_q4_group')
    if group is None or group._layers() is None:
        return None
    if not all(_plain_no_bias(l) and l.scales.dtype == torch.float16 for l in (gate, up, down)):
        return None
    info = quant_hip._layer_info(down.qweight, down.qzeros, down.scales, down.g_idx, down.groupsize)
    if info.plan is not None or info.gemv_gidx is not None:
        return None
    return ((gate.qweight, gate.qzeros, gate.scales), (up.qweight, up.qzeros, up.scales),
            (down.qweight, down.qzeros, down.scales), int(gate.groupsize), gate.in_features, gate.out_features, down.out_features)


def _adapters_off(layer):
    return None if type(layer) is Autograd4bitQuantLinear else getattr(layer, 'disable_adapters', None)


def _mlp_decode_forward(mlp, x):
    """LlamaMLP.forward with the decode step (up to 16 rows, no grad, fp16) as one launch (quant_hip.mlp_decode: gate, up,
    silu(gate) * up and down) or two (quant_hip.mlp_rows); everything else goes to the block's own forward.  What the step
    needs of the three layers is looked up once and kept while their buffers, adapters and bias switches stay the same objects / values."""
    quant_hip = matmul_utils_4bit.quant_hip
    d = mlp.__dict__
    if (not torch.is_grad_enabled() and x.dtype == torch.float16 and x.is_cuda and autograd_4bit.backend == 'cuda'
            and matmul_utils_4bit.use_new and matmul_utils_4bit.auto_switch):
        cached = d.get('_q4_mlp_args')
        mods = mlp._modules
        gate, up, down = mods['gate_proj'], mods['up_proj'], mods['down_proj']
        group = gate.__dict__.get('_q4_group')
        layers = None if group is None else group._layers()  # the same list as long as nothing about gate and up changed
        b0, b1, b2 = gate._buffers.get('bias'), up._buffers.get('bias'), down._buffers.get('bias')
        flags = (-1 if b0 is None else b0._version, -1 if b1 is None else b1._version, -1 if b2 is None else b2._version,
                 gate.disable_bias, up.disable_bias, down.disable_bias, _adapters_off(gate), _adapters_off(up), _adapters_off(down))
        if (cached is None or cached[0] is not layers or cached[1] is not b0 or cached[2] is not b1 or cached[3] is not b2
                or cached[4] != flags or (cached[5] is not None and not _same_layer(down, cached[6]))):
            args = _mlp_decode_args(mlp)
            cached = d['_q4_mlp_args'] = (layers, b0, b1, b2, flags, args, None if args is None else _layer_key(down))
        args = cached[5]
        if args is not None and x.shape[-1] == args[4]:
            rows = x.numel() // args[4]
            if (1 <= rows <= min(int(matmul_utils_4bit.auto_switch_thd), quant_hip.MAX_GEMV_ROWS)
                    and quant_hip.mlp_decode_applicable(rows, args[4], args[5], args[3]) and _is_silu(mods.get('act_fn') if 'act_fn' in mods else getattr(mlp, 'act_fn', None))
                    and (rows <= mlp_decode_max_rows or (d.get('_q4_mlp_gated') and _steps_unobserved(mlp)))):
                faster = quant_hip.mlp_rows_is_faster(rows, args[4], args[5])
                step = quant_hip.mlp_rows_prepared if faster or rows > mlp_decode_max_rows else quant_hip.mlp_decode_prepared
                return step(x, args[0], args[1], args[2], args[3], tuple(x.shape[:-1]) + (args[6],))
    if x.is_cuda and d.get('_q4_mlp_gated') and _act_unobserved(mlp):
        return _gated_rows_forward(mlp, x)
    return d['_q4_mlp_forward'](x)


def make_fused_mlp(model, is_v1_model=False, concatenate=False, fuse_decode_step=True):
    """One launch for gate_proj / up_proj of every MLP block (model_attn_mlp_patch.py:163-247; the reference's Triton
    fused-MLP kernel is replaced by one launch over both projections followed by the block's own activation).  In place
    by default; then, with `fuse_decode_step` and a SiLU block of three 4-bit layers of the same group size, the block's
    forward runs the whole decode step (gate, up, silu(gate) * up, down) as one launch or two."""
    if is_v1_model:
        raise NotImplementedError("v1 (fp zeros) layers are not fused")
    names = ("gate_proj", "up_proj")
    count = 0
    for m in list(model.modules()):
        if all(hasattr(m, n) for n in names + ("down_proj",)):
            if concatenate:
                count += bool(_fuse_children(m, names, "gate_up_proj"))
                continue
            group = _group_children(m, names)
            count += group is not None
            down = m.down_proj
            if (group is not None and fuse_decode_step and _is_silu(getattr(m, 'act_fn', None))
                    and isinstance(down, Autograd4bitQuantLinear) and down.bits == 4 and not down.is_v1_model
                    and down.groupsize == m.gate_proj.groupsize and down.in_features == m.gate_proj.out_features
                    and down.out_features == m.gate_proj.in_features and '_q4_mlp_forward' not in m.__dict__):
                import types
                m.__dict__['_q4_mlp_gated'] = _is_gated_forward(m.forward)
                m.__dict__['_q4_mlp_forward'] = m.forward                # the block's own (bound) forward
                m.__dict__['forward'] = types.MethodType(_mlp_decode_forward, m)
    if concatenate and torch.cuda.is_available():
        torch.cuda.empty_cache()
    return count


def _read_adapter_state(lora_path):
    """Tensors of a saved adapter; only loaders that execute nothing from the file."""
    st = os.path.join(lora_path, "adapter_model.safetensors")
    if os.path.exists(st):
        from safetensors.torch import load_file
        return load_file(st)
    return torch.load(os.path.join(lora_path, "adapter_model.bin"), map_location="cpu", weights_only=True)


_ADAPTER_KEY = re.compile(r"^(?:base_model\.model\.)?(.*)\.(q_proj|k_proj|v_proj)\.lora_([AB])(?:\.[^.]+)?\.weight$")


def inject_lora_layers(model, lora_path, device='cuda', dtype=torch.float16):
    """Loads the adapter saved under `lora_path` (adapter_config.json + adapter_model.safetensors / .bin) onto the
    attention projections.  Same call as the reference's (model_attn_mlp_patch.py:283-335: q_proj and v_proj adapters,
    scaling = lora_alpha / r, a second call replaces the adapter of the first); k_proj adapters are accepted as well.
    On a block fused with `concatenate=True` the adapters become one block-structured adapter on `qkv_proj`; on a block
    grouped in place (or not fused at all) every projection named in the file becomes a LoRA layer of its own that
    shares the projection's packed tensors and keeps its place in the group.  Returns the injected layers."""
    from .models import Linear4bitLt, _share_quant_tensors
    print('Device: {}, dtype: {}'.format(device, dtype))
    with open(os.path.join(lora_path, 'adapter_config.json'), 'r') as fh:
        cfg = json.load(fh)
    scaling = cfg['lora_alpha'] / cfg['r']

    per_block = {}                                           # attention module path -> {(proj, 'A'|'B'): tensor}
    for key, tensor in _read_adapter_state(lora_path).items():
        m = _ADAPTER_KEY.match(key)
        if m is not None:
            per_block.setdefault(m.group(1), {})[(m.group(2), m.group(3))] = tensor

    def lora_layer(base, a, b):
        # lora_alpha = scaling * rank keeps the layer's own scaling (lora_alpha / r) at the saved adapter's value
        rank = a.shape[0]
        layer = Linear4bitLt('default', base.in_features, base.out_features, base.groupsize, False,
                             r=rank, lora_alpha=scaling * rank, lora_dropout=0.0)
        _share_quant_tensors(layer, base)
        layer.disable_bias = base.disable_bias
        layer.lora_A['default'].weight = nn.Parameter(a, requires_grad=False)
        layer.lora_B['default'].weight = nn.Parameter(b, requires_grad=False)
        layer.is_lora_injected = True
        return layer

    modules = dict(model.named_modules())
    injected = []
    for path, parts in per_block.items():
        attn = modules.get(path)
        if attn is None:
            raise ValueError(f'the adapter names {path}, which the model does not have')
        projs = {n: getattr(attn, n, None) for n in ('q_proj', 'k_proj', 'v_proj')}
        present = [n for n in projs if (n, 'A') in parts and (n, 'B') in parts]
        fused = getattr(attn, 'qkv_proj', None)
        if isinstance(fused, Autograd4bitQuantLinear):       # concatenated block: one block-structured adapter
            rank = sum(parts[(n, 'A')].shape[0] for n in present)
            a_cat = torch.cat([parts[(n, 'A')].to(device=device, dtype=dtype) for n in present], dim=0)
            b_blk = torch.zeros(fused.out_features, rank, device=device, dtype=dtype)
            col = 0
            for n in present:
                b = parts[(n, 'B')].to(device=device, dtype=dtype)
                b_blk[projs[n]._start:projs[n]._stop, col:col + b.shape[1]] = b
                col += b.shape[1]
            layer = lora_layer(fused, a_cat, b_blk)
            attn.qkv_proj = layer
            projs['q_proj']._group.layer = layer
            injected.append(layer)
            continue
        for n in present:                                    # projections on their own tensors
            base = projs[n]
            if not isinstance(base, Autograd4bitQuantLinear) or base.is_v1_model:
                raise ValueError(f'{path}.{n} is not a 4-bit (v2) layer')
            layer = lora_layer(base, parts[(n, 'A')].to(device=device, dtype=dtype), parts[(n, 'B')].to(device=device, dtype=dtype))
            group = base.__dict__.get('_q4_group')
            setattr(attn, n, layer)
            if group is not None:
                group.replace(base, layer)
            injected.append(layer)
    print('Lora Injected.')
    return injected
