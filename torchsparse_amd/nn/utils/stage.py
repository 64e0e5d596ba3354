"""Stages: runs of convolutions (with their norms, activations and shortcuts) that one native call
carries out (``csrc/native``).

A network is a tree of small modules, and a sparse convolution through that tree costs the host several
times its launch (module calls, cache look-ups; in training six autograd nodes and a dozen launches made
from Python).  A stage is compiled once from the
modules it stands for: the list of its operations, the parameters they read, and the geometries of the
kernel maps they need.  A call then fetches or builds the maps - the part that is Python's, and that
overlaps with what the device is doing - and hands the rest to one native call; in training the stage
is one autograd node.

``run(module, x)`` answers None for anything a stage does not stand for - hooks on one of the modules, inference in
the dataflows of pair lists, mixed types, norms in evaluation mode - and the caller goes through the modules then.  Results are
those of the modules (in training up to the rounding of what no longer goes through memory between them)."""
import weakref
from typing import List, Optional, Tuple

import torch
from torch import nn
from torch.nn.modules import module as _torch_module

from ...tensor import SparseTensor
from ...utils import make_ntuple
from ..functional.conv import conv_config as _cfg
from ..functional.conv.conv import kernel_map
from ..functional.conv.conv_mode import get_conv_mode
from ..functional.conv.kmap import transpose_kernel_map

__all__ = ["run", "call", "enabled", "forget"]

enabled = True  # False: every module is called on its own

_plans = weakref.WeakKeyDictionary()  # module -> {(training, placed): _Plan or None}


class _Unfit(Exception):
    """The modules are not what a stage stands for."""


class _Plan:
    __slots__ = ("native", "slots", "modules", "members", "convs", "training", "cin", "lead", "out_level", "config")

    def current(self) -> bool:
        """Whether the modules still are what the plan was compiled from: the same parameters and buffers, no hooks."""
        for m in self.modules:
            if (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                    or m.training is not self.training):
                return False
        for table, name, value in self.members:
            if table[name] is not value:
                return False
        for conv, config, activation in self.convs:
            if conv._config is not config or conv.activation != activation:
                return False
        return True


def _no_global_hooks() -> bool:
    t = _torch_module
    return not (t._global_forward_hooks or t._global_forward_pre_hooks or t._global_backward_hooks
                or t._global_backward_pre_hooks)


class _Builder:
    def __init__(self, training: bool):
        from ..modules import BatchNorm, Conv3d, ReLU
        self.Conv3d, self.BatchNorm, self.ReLU = Conv3d, BatchNorm, ReLU
        self.training = training
        self.ops, self.params, self.slots, self.modules, self.members = [], [], [], [], []
        self.index = {}
        self.buffers, self.level, self.config = 1, 0, None

    def param(self, module, name) -> int:
        value = module._parameters[name]
        if value is None:
            return -1
        if value.is_inference() or not value.is_contiguous():
            raise _Unfit
        self.members.append((module._parameters, name, value))
        if id(value) not in self.index:
            self.index[id(value)] = len(self.params)
            self.params.append(value)
        return self.index[id(value)]

    def see(self, module) -> None:
        self.modules.append(module)

    def conv(self, conv, src: int, norm=None, relu: bool = False, residual: int = -1) -> int:
        """Appends act(norm(conv(src)) + residual); returns the buffer of the result."""
        if type(conv) is not self.Conv3d or conv.generative or (self.ops and conv._config is not self.config):
            raise _Unfit
        self.config = conv._config
        self.see(conv)
        kernel = conv._parameters["kernel"]
        if conv.activation not in (None, "relu") or (self.training and (conv.activation or conv.bias is not None)):
            raise _Unfit
        if not self.training:
            relu = relu or conv.activation == "relu"
        stride, dilation = conv.stride, make_ntuple(conv.dilation, ndim=3)
        pointwise = kernel.dim() == 2
        if pointwise and (conv.kernel_size != (1, 1, 1) or stride != (1, 1, 1) or dilation != (1, 1, 1)):
            raise _Unfit
        if not pointwise and conv.kernel_size == (1, 1, 1) and stride == (1, 1, 1) and dilation == (1, 1, 1):
            raise _Unfit
        after = self.level
        if conv.transposed:
            after = self.level - 1
        elif stride != (1, 1, 1):
            after = self.level + 1
        slot = (self.level, after, conv.kernel_size, stride, dilation, conv.transposed, conv.padding, pointwise)
        wide = conv.out_channels >= 128 or kernel.dtype == torch.float32
        at = next((i for i, s in enumerate(self.slots) if s[0] == slot), None)
        if at is None:
            at = len(self.slots)
            self.slots.append([slot, None, 0])
        if not pointwise and conv.kernel_volume >= 27:
            most = self.slots[at][1]  # (channels by which a map's form is decided)
            if wide and (most is None or conv.in_channels * conv.out_channels > most[1] * most[2]):
                self.slots[at][1] = (conv.kernel_volume, conv.in_channels, conv.out_channels)
            self.slots[at][2] += 1
        self.level = after
        dst = self.buffers
        self.buffers += 1
        if conv.kernel.shape[-1] != conv.out_channels or conv.kernel.shape[-2] != conv.in_channels:
            raise _Unfit
        self.ops.append(((src, dst, residual, at, bool(conv.transposed), relu, self.param(conv, "kernel"),
                          self.param(conv, "bias"), conv.kernel_volume, conv.in_channels, conv.out_channels), norm))
        return dst

    # -- the modules a stage is made of

    def sequence(self, modules: List[nn.Module], src: int, residual: int = -1, relu_after: bool = False) -> int:
        """The modules one after the other; ``residual`` / ``relu_after``: what follows the last of them."""
        modules = [m for m in modules if m.__class__ is not nn.Identity]
        i = 0
        while i < len(modules):
            m = modules[i]
            if isinstance(m, self.Conv3d):
                norm, relu, used = None, False, 1
                if self.training:
                    if i + 1 >= len(modules) or type(modules[i + 1]) is not self.BatchNorm:
                        raise _Unfit
                    norm, used = modules[i + 1], 2
                    if i + 2 < len(modules) and type(modules[i + 2]) is self.ReLU:
                        relu, used = True, 3
                        self.see(modules[i + 2])
                last = i + used == len(modules)
                src = self.conv(m, src, norm, relu or (last and relu_after), residual if last else -1)
                i += used
            else:
                if residual >= 0 and i + 1 == len(modules):
                    raise _Unfit
                src = self.module(m, src)
                i += 1
        return src

    def module(self, m: nn.Module, src: int) -> int:
        from ...backbones.detection import SparseBasicBlock
        from ...backbones.modules.blocks import SparseResBlock, _Chain
        from .fuse import FoldedSequential
        if isinstance(m, self.Conv3d):
            return self.sequence([m], src)
        if m.__class__ is nn.Identity:
            return src
        if type(m).forward in (nn.Sequential.forward, FoldedSequential.forward, _Chain.forward):
            self.see(m)
            return self.sequence(list(m._modules.values()), src)
        if type(m) is SparseResBlock:
            self.see(m)
            main, shortcut = m.main, m.shortcut
            self.see(main)
            if not self.training and not getattr(m, "_fused_tail", False):
                raise _Unfit
            if type(main).forward not in (nn.Sequential.forward, FoldedSequential.forward):
                raise _Unfit
            side = src
            if shortcut.__class__ is not nn.Identity:
                level = self.level
                side = self.module(shortcut, src)
                self.level = level
            if self.training:
                if type(m.relu) is not self.ReLU:
                    raise _Unfit
                self.see(m.relu)
            # (in inference form the last convolution carries the activation itself)
            return self.sequence(list(main), src, residual=side, relu_after=self.training)
        if type(m) is SparseBasicBlock and not self.training and getattr(m, "_fused_tail", False):
            self.see(m)
            return self.conv(m.conv2, self.conv(m.conv1, src), residual=src)
        raise _Unfit

    def finish(self, out: int):
        from ... import backend
        if not self.ops or out != self.ops[-1][0][1]:
            raise _Unfit
        norms = {}
        for op, norm in self.ops:  # (every parameter is known before the native stage is made)
            if norm is not None:
                self.see(norm)
                gamma, beta = self.param(norm, "weight"), self.param(norm, "bias")
                if norm.momentum is None or not norm.training or (gamma < 0) != (beta < 0) or norm.num_features != op[10]:
                    raise _Unfit
                for name in ("running_mean", "running_var", "num_batches_tracked"):
                    self.members.append((norm._buffers, name, norm._buffers.get(name)))
                track = norm.track_running_stats
                norms[op[1]] = (gamma, beta, *(norm._buffers.get(k) if track else None
                                               for k in ("running_mean", "running_var")),
                                norm._buffers.get("num_batches_tracked"), float(norm.momentum), float(norm.eps))
        dtypes = {p.dtype for p in self.params}
        if len(dtypes) != 1 or any(not p.is_cuda for p in self.params):
            raise _Unfit
        per = 16 // next(iter(dtypes)).itemsize
        native = backend.native().Stage(self.params, self.buffers)
        for op, norm in self.ops:
            native.add(*op)
            if norm is None:
                continue
            gamma, beta, mean, var, batches, momentum, eps = norms[op[1]]
            channels = op[10]
            if channels % per or channels // per > 256 or any(
                    t is not None and (t.dtype not in dtypes or not t.is_contiguous() or not t.is_cuda)
                    for t in (mean, var)):
                raise _Unfit
            if batches is not None and (batches.dtype != torch.int64 or not batches.is_cuda):
                raise _Unfit
            native.norm(*norms[op[1]])
        plan = _Plan()
        plan.native, plan.training = native, self.training
        plan.slots = tuple((tuple(s[0]), s[1], s[2]) for s in self.slots)
        plan.modules, plan.members = tuple(self.modules), tuple(self.members)
        plan.convs = tuple((m, m._config, m.activation) for m in self.modules if type(m) is self.Conv3d)
        plan.lead = self.params[0]
        plan.cin = self.ops[0][0][9]
        plan.out_level = self.level
        plan.config = self.config
        return plan


def _compile(modules: Tuple[nn.Module, ...], training: bool) -> Optional[_Plan]:
    try:
        b = _Builder(training)
        out = 0
        if training and len(modules) == 1 and type(modules[0]) is b.Conv3d:
            return b.finish(b.conv(modules[0], 0))  # (a layer on its own needs no norm behind it)
        for m in modules:
            out = b.module(m, out)
        return b.finish(out)
    except (_Unfit, KeyError, AttributeError):
        return None


def _plan_of(owner: nn.Module, modules: Tuple[nn.Module, ...], key) -> Optional[_Plan]:
    table = _plans.get(owner)
    if table is None:
        table = _plans[owner] = {}
    plan = table.get(key, table)  # (the table itself: not compiled yet)
    if plan is not table and plan is not None and not plan.current():
        plan = table  # (parameters or buffers were replaced, or hooks were added)
    if plan is table:
        plan = table[key] = _compile(modules, key[0])
        if plan is not None and not plan.current():
            return None  # (hooks: the plan waits until they are gone)
    return plan


def forget() -> None:
    """Every plan is made anew: layers were given other configurations, or were fused."""
    _plans.clear()


def _native_map(backend, kmap, transposed: bool):
    handle = dict.get(kmap, "_native")
    if handle is None:
        omap = kmap["out_in_map"]
        n_in, n_out = kmap["sizes"]
        odd = all(k % 2 == 1 for k in kmap["kernel_size"])
        handle = backend.native().KernelMap(omap.shape[1], n_in, n_out, bool(kmap["subm"] and kmap["distinct"] and odd),
                                            omap, kmap.get("out_in_map_t"))
        kmap["_native"] = handle
    elif transposed and not handle.has_transposed:
        handle.set_transposed(kmap["out_in_map_t"])
    return handle


_LISTS = {_cfg.Dataflow.GatherScatter: 1, _cfg.Dataflow.FetchOnDemand: 2}


def _pair_lists(handle, kmap, form: int) -> bool:
    """Whether the map has the pair lists of that dataflow; the native map has them then, too."""
    if handle.lists == 0:
        nbmaps, nnz = kmap["nbmaps"], kmap.get("nnz")
        if nbmaps is None or nbmaps.dtype != torch.int32 or nbmaps.shape != ((nnz, 2) if form == 1 else (2, nnz)):
            return False
        centered = bool(kmap["subm"]) and kmap["out_in_map"].shape[1] % 2 == 1
        handle.set_lists(form == 2, nbmaps, kmap["nbaddrs"], kmap["qnbaddrs"], int(kmap["qmapsize"]),
                         kmap["output_mask"], kmap["input_mask"], centered)
    return handle.lists == form


def run(owner: nn.Module, x: SparseTensor, modules: Optional[Tuple[nn.Module, ...]] = None, place=None, also=None):
    """What ``owner`` (or the ``modules`` it stands for, one after the other) makes of ``x``, by one native
    call; None where it has to be called itself.  ``place`` = (buffer, first column): the first convolution's
    result goes there, and the buffer is what the next one reads.  ``also`` = (columns, first column): the
    result a second time in a new buffer of that many columns, and (result, buffer) is returned."""
    feats = x.feats
    if not (enabled and feats.is_cuda):
        return None
    training = owner.training
    from ... import backend
    grad = torch.is_grad_enabled()
    if (training != grad and (training or feats.requires_grad)) or backend._pin_sinks or not _no_global_hooks():
        return None
    if training and (place is not None or also is not None):
        return None
    plan = _plan_of(owner, modules or (owner,), (training, place is not None))
    if plan is None:
        return None
    if not training and grad and any(p.requires_grad for p in plan.native.params):
        return None
    if feats.dtype != plan.lead.dtype or not feats.is_contiguous() or feats.device != plan.lead.device:
        return None
    if feats.shape[1] != plan.cin or feats.shape[0] < (2 if training else 1):
        return None
    config = plan.config or _cfg.get_global_conv_config()
    if config is None:
        config = _cfg._shared_default_config(get_conv_mode())
    lists = config["dataflow"] != _cfg.Dataflow.ImplicitGEMM
    if config["ifsort"] or (lists and (not training or config["dataflow"] not in _LISTS)):
        return None
    force = config.get("pair_segments")
    caches = x._caches
    strides = {0: x.stride}
    levels = caches.cmaps
    if x.stride not in levels:
        levels[x.stride] = (x.coords, x.spatial_range)
    maps, segments = [], False
    for (level, after, kernel_size, stride, dilation, transposed, padding, pointwise), wide, uses in plan.slots:
        here = strides[level]
        coords, spatial_range = (x.coords, x.spatial_range) if level == 0 else levels[here]
        if pointwise:
            maps.append(backend.native_identity(coords.shape[0]))
            continue
        if transposed:
            fine = tuple(here[a] // stride[a] for a in range(3))
            strides[after] = fine
            kmap = caches.kmaps.get((fine, kernel_size, stride, dilation))
            if kmap is None or fine not in levels:
                return None  # (the module's own call raises what there is to raise)
            if not lists:
                transpose_kernel_map(kmap, False)
        else:
            if after != level:
                strides[after] = tuple(here[a] * stride[a] for a in range(3))
            key = (here, kernel_size, stride, dilation)
            kmap = caches.kmaps.get(key)
            if kmap is None:
                kmap = kernel_map(caches, key, coords, coords.shape[0], padding, spatial_range, config, training)
            if strides[after] not in levels:
                levels[strides[after]] = (kmap["coords"], kmap["spatial_range"])
        if kmap["sizes"][0] == 0 or kmap["sizes"][1] < (2 if training else 1):
            return None
        dict.setdefault(kmap, "kernel_size", kernel_size)
        handle = _native_map(backend, kmap, transposed and not lists)
        if lists and not _pair_lists(handle, kmap, _LISTS[config["dataflow"]]):
            return None
        if wide is not None and not transposed and (not lists or kmap["subm"]):
            coarse = levels.get(tuple(2 * s for s in here))
            segments = backend.native_segments(handle, feats, wide, kmap, force, coarse and coarse[0]) or segments
        if uses and not transposed:  # (in training the input gradient of a submanifold layer is a second use)
            uses = (0 if lists else uses) + (uses if training and kmap["subm"] else 0)
            if uses:
                backend.native_grouped(handle, kmap, uses)
        maps.append(handle)
    out_stride = strides[plan.out_level]
    out_coords, out_range = (x.coords, x.spatial_range) if plan.out_level == 0 else levels[out_stride]
    if training:
        if backend._region_calls:
            backend.flush_launches()
        y = plan.native.train(feats, maps, segments, lists, backend.group_min_rows)
        return SparseTensor._make(y, out_coords, out_stride, out_range, caches)
    pending = backend.pending_calls()
    if also is not None:
        buffer = feats.new_empty(out_coords.shape[0], also[0])
        also = (buffer, also[1])
    y = plan.native.run(feats, maps, segments, backend.group_min_rows, -1 if place is None else 0, place, also, pending)
    if pending is not None:
        backend.keep_pending(pending)
    out = SparseTensor._make(y, out_coords, out_stride, out_range, caches)
    return out if also is None else (out, buffer)


def call(module: nn.Module, x: SparseTensor) -> SparseTensor:
    """``module(x)``, as a stage where it is one."""
    y = run(module, x)
    return module(x) if y is None else y
