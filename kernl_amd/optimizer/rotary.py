"""Fuse the rotary position embedding of Hugging Face decoders into one kernel per tensor.

`apply_rotary_pos_emb` traces to, per tensor,

    x * cos + cat((-x[..., D/2:], x[..., :D/2]), dim=-1) * sin

i.e. two slices, a negation, a concatenation, two multiplications and an addition: seven element-wise kernels and six
intermediate tensors for what is one read and one write of x.  The reference removes the same overhead in its Llama
experiment by rotating inside the query/key projection (experimental/llama-v2/kernel/fused_kernel_proj_qkv.py:69-100).
The slice bound is a literal that differs per model, so the sub-graph is matched by walking it rather than by
`replace_pattern`.  The tables, which trace to nine kernels per forward, become one launch (`fuse_rotary_tables`).
"""
import operator

import torch
from torch.fx import Node

from kernl_amd.implementations.rotary import rotary_forward, rotary_tables


def rotary_wrapper(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    return rotary_forward(x, cos, sin)


def rotary_tables_wrapper(inv_freq: torch.Tensor, positions: torch.Tensor, scale: float, dtype: torch.dtype):
    return rotary_tables(inv_freq, positions, scale, dtype)


torch.fx.wrap("rotary_wrapper")
torch.fx.wrap("rotary_tables_wrapper")

_MUL = (operator.mul, torch.mul)
_ADD = (operator.add, torch.add)
_NEG = (operator.neg, torch.neg)


def _is_call(node, targets) -> bool:
    return isinstance(node, Node) and node.op == "call_function" and node.target in targets


def _last_dim_slice(node):
    """(source, start, stop) for `source[..., start:stop]`, else None."""
    if not _is_call(node, (operator.getitem,)) or len(node.args) != 2:
        return None
    source, index = node.args
    if not (isinstance(index, tuple) and len(index) == 2 and index[0] is Ellipsis and isinstance(index[1], slice)):
        return None
    sl = index[1]
    if sl.step not in (None, 1):
        return None
    return source, sl.start, sl.stop


def _rotate_half_source(cat: Node):
    """x and the split point h if `cat` is cat((-x[..., h:], x[..., :h]), dim=-1), else None."""
    if not _is_call(cat, (torch.cat,)) or not cat.args:
        return None
    operands = cat.args[0]
    dim = cat.kwargs.get("dim", cat.args[1] if len(cat.args) > 1 else 0)
    if dim != -1 or not isinstance(operands, (list, tuple)) or len(operands) != 2:
        return None
    neg, low = operands
    if not _is_call(neg, _NEG):
        return None
    high_slice, low_slice = _last_dim_slice(neg.args[0]), _last_dim_slice(low)
    if high_slice is None or low_slice is None:
        return None
    (xa, start_a, stop_a), (xb, start_b, stop_b) = high_slice, low_slice
    if xa is not xb or stop_a is not None or start_b not in (None, 0) or not isinstance(start_a, int) or start_a != stop_b:
        return None
    return xa, start_a


def fuse_rotary_embedding(gm: torch.fx.GraphModule):
    changed = False
    for add in list(gm.graph.nodes):
        if not _is_call(add, _ADD) or len(add.args) != 2 or add.kwargs:
            continue
        for direct, rotated in (add.args, add.args[::-1]):
            if not (_is_call(direct, _MUL) and _is_call(rotated, _MUL)):
                continue
            found = None
            for cat, sin in (rotated.args, rotated.args[::-1]):
                src = _rotate_half_source(cat) if isinstance(cat, Node) else None
                if src is None or not isinstance(sin, Node):
                    continue
                x, half = src
                for xx, cos in (direct.args, direct.args[::-1]):
                    if xx is x and isinstance(cos, Node):
                        found = (x, cos, sin, half)
                        break
                if found:
                    break
            if not found:
                continue
            x, cos, sin, half = found
            # the split must be at the middle of the feature dimension: known only when the tracer recorded shapes
            example = x.meta.get("example_value")
            if example is None or example.dim() != 4 or example.shape[-1] != 2 * half:
                continue
            with gm.graph.inserting_before(add):
                fused = gm.graph.call_function(rotary_wrapper, (x, cos, sin))
            fused.meta = dict(add.meta)
            add.replace_all_uses_with(fused)
            changed = True
            break
    if changed:
        gm.graph.eliminate_dead_code()
        gm.graph.lint()
        gm.recompile()


def _is_method(node, name) -> bool:
    return isinstance(node, Node) and node.op == "call_method" and node.target == name


def _example(node):
    value = node.meta.get("example_value") if isinstance(node, Node) else None
    return value if isinstance(value, torch.Tensor) else None


def _converted_to(node):
    """The dtype if `node` is x.to(dtype) — alone or with x's own device — or x.float(), else None."""
    if _is_method(node, "float") and len(node.args) == 1 and not node.kwargs:
        return torch.float32
    if not _is_method(node, "to"):
        return None
    source = _example(node.args[0])
    wanted = list(node.args[1:]) + [node.kwargs[k] for k in node.kwargs if k in ("dtype", "device")]
    dtypes = [w for w in wanted if isinstance(w, torch.dtype)]
    others = [w for w in wanted if not isinstance(w, torch.dtype)]
    if len(dtypes) != 1 or set(node.kwargs) - {"dtype", "device"} or source is None:
        return None
    if any(not isinstance(w, (str, torch.device)) or torch.device(w) != source.device for w in others):
        return None
    return dtypes[0]


def _before_float32(node, exact):
    """What `node` converts to float32, through as many conversions as there are, if that is of a dtype in `exact`."""
    while _converted_to(node) is torch.float32:
        source = _example(node.args[0])
        if source is None or source.dtype not in exact:
            break
        node = node.args[0]
    return node


def fuse_rotary_tables(gm: torch.fx.GraphModule):
    """`a = (inv_freq @ positions).transpose(1, 2); e = cat((a, a), -1); (e.cos() * s).to(dtype), (e.sin() * s).to(dtype)`, the
    product of inner size one in float32 and nothing else reading e, becomes one `rotary_tables_wrapper` call, which takes the frequencies
    and whole positions before their conversion to float32.  A whole zero added to the `arange` of the positions goes too."""
    changed = False
    for cat in list(gm.graph.nodes):
        if not _is_call(cat, (torch.cat,)) or not cat.args or cat.kwargs.get("dim", cat.args[1] if len(cat.args) > 1 else 0) != -1:
            continue
        parts = cat.args[0]
        if not isinstance(parts, (list, tuple)) or len(parts) != 2 or parts[0] is not parts[1] or not _is_method(parts[0], "transpose"):
            continue
        turned = parts[0]
        product = turned.args[0]
        if tuple(turned.args[1:]) not in ((1, 2), (2, 1)) or turned.kwargs or not _is_call(product, (operator.matmul, torch.matmul, torch.bmm)):
            continue
        left, right = (product.args + (None, None))[:2]
        lv, rv, ev = _example(left), _example(right), _example(cat)
        if any(v is None or v.dim() != 3 or v.dtype != torch.float32 for v in (lv, rv, ev)) or lv.shape[2] != 1 or lv.shape[1] < 1:
            continue
        ends = {}
        for user in cat.users:
            name = next((n for n in ("cos", "sin") if _is_method(user, n) or _is_call(user, (getattr(torch, n),))), None)
            if name is None or name in ends:
                break
            end, scale, dtype = user, 1.0, torch.float32
            after = next(iter(end.users)) if len(end.users) == 1 else None
            if _is_call(after, _MUL) and len(after.args) == 2 and not after.kwargs and isinstance(after.args[1], (int, float)):
                end, scale = after, float(after.args[1])
                after = next(iter(end.users)) if len(end.users) == 1 else None
            if isinstance(after, Node) and _converted_to(after) in (torch.float16, torch.bfloat16, torch.float32):
                end, dtype = after, _converted_to(after)
            ends[name] = (end, scale, dtype)
        if len(ends) != len(cat.users) or set(ends) != {"cos", "sin"} or ends["cos"][1:] != ends["sin"][1:]:
            continue
        _, scale, dtype = ends["cos"]
        inv_freq = _before_float32(left, (torch.float16, torch.bfloat16, torch.float32))
        positions = _before_float32(right, (torch.int64, torch.float32))
        with gm.graph.inserting_after(cat):
            tables = gm.graph.call_function(rotary_tables_wrapper, (inv_freq, positions, scale, dtype))
        with gm.graph.inserting_after(tables):
            outs = [gm.graph.call_function(operator.getitem, (tables, i)) for i in (0, 1)]
        for out, name in zip(outs, ("cos", "sin")):
            out.meta = dict(ends[name][0].meta)
            ends[name][0].replace_all_uses_with(out)
        changed = True
        for node in list(gm.graph.nodes):
            start = node.args[0] if _is_call(node, _ADD) and len(node.args) == 2 and not node.kwargs else None
            if (_is_call(start, (torch.arange,)) and len(start.users) == 1 and type(node.args[1]) is int and node.args[1] == 0
                    and _example(start) is not None and _example(start).dtype == torch.int64):
                node.replace_all_uses_with(start)
    if changed:
        gm.graph.eliminate_dead_code()
        gm.graph.lint()
        gm.recompile()
