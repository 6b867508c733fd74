"""Attention written with matrix products and a softmax, found in a traced graph.

``softmax(q k^T c) v`` over per-head arrays ``(H, n, d)`` arrives from the trace as two batched products with a softmax
between them, wrapped in views, permutations and copies that differ with the way the model spells it (``matmul``, ``einsum``,
``bmm``, one head or several).  ``fuse_attention`` replaces such a group by ONE equation, which the attention rule evaluates
(``multi_head_self_attention``, the rule the reference registers for its attention kernel,
folx/experimental/pallas/attention/__init__.py:45); a mask, a dropout or a second reader anywhere between the two products
leaves the group as it is.

Every view on the way is followed as a permutation of flat indices, so the pattern does not depend on which views were used."""

from __future__ import annotations

import math

import torch

aten = torch.ops.aten

# views and copies: the result holds the operand's entries in some order
_INDEXING = {aten.view.default, aten._unsafe_view.default, aten.reshape.default, aten.transpose.int, aten.permute.default,
             aten.t.default, aten.expand.default, aten.unsqueeze.default, aten.squeeze.dim, aten.squeeze.dims,
             aten.squeeze.default, aten.clone.default, aten.contiguous.default, aten.alias.default}
_PRODUCTS = {aten.bmm.default, aten.mm.default}
# What the attention kernels take; beyond, the products and the softmax are the rule anyway.  Replayed calls of 280 random sizes (1 to 4096
# walkers, 1 to 8 heads, d = 4 .. 64): 0.42 of the time of the products apart in the geometric mean.  Two took longer, single walkers of more than 16
# positions, where one workgroup a head walks all Jacobian rows (n = 21, d = 20: 209 us for 172); a line there would make a walker's
# result depend on its batch.
_MAX_N = _MAX_D = 64
_MAX_ENTRIES = 1 << 22            # of an operand whose views are followed


def attention(q, k, v):
    """What a fused group computes: ``softmax(q k^T) v`` for ``(n, H, d)``."""
    p = torch.softmax(torch.einsum('ihd,jhd->hij', q, k), dim=-1)
    return torch.einsum('hij,jhd->ihd', p, v)


def _shape(node):
    val = node.meta.get('val')
    return tuple(val.shape) if isinstance(val, torch.Tensor) and val.dtype == torch.float32 else None


def _replay(node, index):
    """The view or copy ``node`` applied to the index array of its operand; None if it repeats entries.  The index is taken in
    its own order first: whether a view exists depends on strides, and those of the array in the trace are others."""
    index = index.contiguous()
    args = [index if a is node.args[0] else a for a in node.args]
    kwargs = {k: a for k, a in node.kwargs.items() if k != 'memory_format'}
    if any(isinstance(a, torch.fx.Node) for a in args):
        return None
    out = node.target(*args, **kwargs)
    return out if out.numel() == index.numel() else None


def _source(node):
    """(source, index): ``node``'s entries as flat indices into ``source``, the first array behind its views."""
    chain = []
    while isinstance(node, torch.fx.Node) and node.op == 'call_function' and node.target in _INDEXING:
        chain.append(node)
        node = node.args[0]
    shape = _shape(node) if isinstance(node, torch.fx.Node) else None
    if shape is None or math.prod(shape) > _MAX_ENTRIES:
        return None
    index = torch.arange(math.prod(shape)).reshape(shape)
    for view in reversed(chain):
        index = _replay(view, index)
        if index is None:
            return None
    return node, index


def _in_order(index, shape):
    """Whether ``index`` of the given shape counts up along it."""
    return tuple(index.shape) == tuple(shape) and bool((index.reshape(-1) == torch.arange(index.numel())).all())


def _scale(node, consts):
    """The factor of ``x * c`` / ``x / c`` with a single number ``c``, else None."""
    if node.target not in (aten.mul.Tensor, aten.mul.Scalar, aten.div.Tensor, aten.div.Scalar) or len(node.args) != 2 or node.kwargs:
        return None
    c = node.args[1]
    if isinstance(c, torch.fx.Node):
        c = consts.get(c)
        if c is None or getattr(c, 'size', 1) != 1 or getattr(c, 'ndim', 0) != 0:
            return None
    c = float(c)
    if node.target in (aten.div.Tensor, aten.div.Scalar):
        return 1.0 / c if c != 0.0 else None    # Python divides by no zero: left to the division itself
    return c


def _down(node, index, used):
    """Follow the single reader of ``node`` through views and copies; yields (last node, index)."""
    while len(node.users) == 1:
        user = next(iter(node.users))
        if user.op != 'call_function' or user.target not in _INDEXING or user.args[0] is not node:
            break
        moved = _replay(user, index)
        if moved is None:
            break
        node, index = user, moved
        used.append(node)
    return node, index


def _operand(node, batched):
    """An operand of a product as (source, index of shape (H, rows, columns))."""
    got = _source(node)
    if got is None:
        return None
    return got[0], got[1] if batched else got[1].unsqueeze(0)


def _match(softmax, consts):
    if softmax.target is not aten._softmax.default or bool(softmax.args[2]):
        return None
    shape = _shape(softmax)
    if shape is None or len(shape) < 2 or int(softmax.args[1]) % len(shape) != len(shape) - 1:
        return None
    # upwards: a factor and views that keep the order, to the first product
    factor, node, inner = 1.0, softmax.args[0], [softmax]
    while isinstance(node, torch.fx.Node) and node.op == 'call_function' and node.target not in _PRODUCTS:
        if len(node.users) != 1:
            return None
        c = _scale(node, consts)
        if c is not None:
            factor *= c
        elif node.target not in _INDEXING:
            return None
        inner.append(node)
        node = node.args[0]
    first = node
    if not isinstance(first, torch.fx.Node) or first.target not in _PRODUCTS or len(first.users) != 1:
        return None
    inner.append(first)
    if math.prod(_shape(first) or ()) != math.prod(shape) or math.prod(shape) > _MAX_ENTRIES:
        return None
    index = torch.arange(math.prod(shape)).reshape(_shape(first))
    for view in reversed(inner[1:-1]):
        if _scale(view, consts) is None:
            index = _replay(view, index)
            if index is None:
                return None
    if not _in_order(index, shape):
        return None
    # downwards: views that keep the order, to the second product
    below = []
    node, index = _down(softmax, torch.arange(math.prod(shape)).reshape(shape), below)
    if len(node.users) != 1:
        return None
    second = next(iter(node.users))
    if second.target not in _PRODUCTS or second.args[0] is not node or second.args[1] is node:
        return None
    batched = first.target is aten.bmm.default
    qs, ks = _operand(first.args[0], batched), _operand(first.args[1], batched)
    vs = _operand(second.args[1], second.target is aten.bmm.default)
    if qs is None or ks is None or vs is None:
        return None
    H, n, d = qs[1].shape
    if (n > _MAX_N or d > _MAX_D or d % 4 != 0 or tuple(ks[1].shape) != (H, d, n) or tuple(vs[1].shape) != (H, n, d)
            or not _in_order(index.reshape(-1), (H * n * n,)) or shape[-1] != n):
        return None
    if any(s[0] in consts for s in (qs, ks, vs)):   # an operand without derivatives: not the attention rule's case
        return None
    return factor, qs, (ks[0], ks[1].transpose(1, 2)), vs, inner + below, second


def _call(gm, target, args, shape):
    node = gm.graph.call_function(target, args)
    node.meta['val'] = torch.empty(shape, device='meta')
    return node


def _heads_inside(gm, source, index):
    """``source`` as ``(n, H, d)``, given the index of its ``(H, n, d)`` form."""
    H, n, d = index.shape
    graph = gm.graph
    if _in_order(index.permute(1, 0, 2), (n, H, d)):
        return graph.call_function(aten.view.default, (source, [n, H, d]))
    if _in_order(index, (H, n, d)):
        return graph.call_function(aten.permute.default, (graph.call_function(aten.view.default, (source, [H, n, d])), [1, 0, 2]))
    return None


def _scaled_weights(gm, source, factor, consts):
    """A product with a constant matrix that nothing else reads, its weights (and bias) times ``factor``; else None."""
    if source.op != 'call_function' or len(source.users) != 1 or source.kwargs:
        return None
    graph = gm.graph
    times = lambda t: graph.call_function(aten.mul.Tensor, (t, factor))     # noqa: E731  (constants: folded with the others)
    if source.target is aten.mm.default and source.args[1] in consts:
        return graph.call_function(aten.mm.default, (source.args[0], times(source.args[1])))
    if source.target is aten.addmm.default and source.args[0] in consts and source.args[2] in consts:
        return graph.call_function(aten.addmm.default, (times(source.args[0]), source.args[1], times(source.args[2])))
    return None


def fuse_attention(gm: torch.fx.GraphModule, consts) -> int:
    """Rewrite ``gm`` in place; ``consts`` are the nodes known to be constant.  Returns the number of groups found."""
    found = 0
    for softmax in [n for n in gm.graph.nodes if n.op == 'call_function' and n.target is aten._softmax.default]:
        got = _match(softmax, consts)
        if got is None:
            continue
        factor, (q, qi), (k, ki), (v, vi), inner, second = got
        forms = [(q, qi), (k, ki), (v, vi)]
        # (n, H, d) or (H, n, d) up to the order of whole axes; anything else stays as it is
        if not all(_in_order(i.permute(1, 0, 2), (i.shape[1], i.shape[0], i.shape[2])) or _in_order(i, i.shape) for _, i in forms):
            continue
        H, n, d = qi.shape
        with gm.graph.inserting_before(second):
            if factor != 1.0:
                scaled = _scaled_weights(gm, q, factor, consts) if q is not k and q is not v else None
                q = scaled if scaled is not None else gm.graph.call_function(aten.mul.Tensor, (q, factor))
            ops = [_heads_inside(gm, node, i) for node, i in ((q, qi), (k, ki), (v, vi))]
            out = _call(gm, attention, tuple(ops), (n, H, d))
            result = _call(gm, aten.permute.default, (out, [1, 0, 2]), (H, n, d))
            if second.target is aten.mm.default:
                result = _call(gm, aten.view.default, (result, [n, d]), (n, d))
        # behind the second product: where the views of its reader bring back the order of (n, H, d), that is read directly
        node, index = second, torch.arange(n * H * d).reshape(n, H, d).permute(1, 0, 2).reshape(_shape(second))
        direct = None
        while True:
            if _in_order(index.reshape(-1), (n * H * d,)):
                direct = node, tuple(index.shape)
            if len(node.users) != 1:
                break
            user = next(iter(node.users))
            if user.op != 'call_function' or user.target not in _INDEXING or user.args[0] is not node:
                break
            index = _replay(user, index)
            if index is None:
                break
            node = user
        if direct is not None:
            with gm.graph.inserting_before(direct[0]):
                view = _call(gm, aten.view.default, (out, list(direct[1])), direct[1])
            direct[0].replace_all_uses_with(view)
        if second.users:
            second.replace_all_uses_with(result)
        found += 1
    if found:
        # the groups' own nodes, and views that only they read
        for node in reversed(list(gm.graph.nodes)):
            if not node.users and node.op == 'call_function' and (
                    node.target in _INDEXING or node.target in _PRODUCTS or node.target in (
                        aten._softmax.default, aten.mul.Tensor, aten.mul.Scalar, aten.div.Tensor, aten.div.Scalar, aten.addmm.default)):
                gm.graph.erase_node(node)
        gm.graph.lint()
    return found
