"""Pytree utilities for argument handling in the transforms.

Same surface as nabla/core/common/pytree.py (tree_flatten / tree_unflatten /
tree_map / tree_leaves / tree_structure / register_pytree_node / PyTreeDef);
no arithmetic lives here.
"""
from __future__ import annotations

from typing import Any, Callable

_REGISTRY: dict[type, tuple[Callable, Callable]] = {}


def register_pytree_node(cls: type, flatten_fn: Callable, unflatten_fn: Callable) -> None:
    """``flatten_fn(obj) -> (children, aux)``; ``unflatten_fn(aux, children) -> obj``."""
    _REGISTRY[cls] = (flatten_fn, unflatten_fn)


class PyTreeDef:
    __slots__ = ("kind", "aux", "children", "num_leaves", "_flat_key", "_hash")

    def __init__(self, kind: Any, aux: Any, children: tuple, num_leaves: int):
        self.kind = kind
        self.aux = aux
        self.children = children
        self.num_leaves = num_leaves
        self._flat_key = self._hash = None

    def _key(self):
        """Nested tuples down to the leaves, made once: compared and hashed without a call of
        Python code per node (a compiled step hashes its arguments' structure at every call)."""
        k = self._flat_key
        if k is None:
            k = self._flat_key = (self.kind, self.aux, tuple([c._key() for c in self.children]))
        return k

    def __eq__(self, other):
        return isinstance(other, PyTreeDef) and self._key() == other._key()

    def __hash__(self):
        h = self._hash
        if h is None:
            try:
                h = hash(self._key())
            except TypeError:  # (an auxiliary value that has no hash)
                h = hash((self.kind, repr(self.aux), self.children))
            self._hash = h
        return h

    def __repr__(self):
        if self.kind is _K_LEAF:
            return "*"
        return f"PyTreeDef({getattr(self.kind, '__name__', self.kind)}, {list(self.children)})"


_K_LEAF = "leaf"
_K_NONE = "none"
_LEAF_DEF = PyTreeDef(_K_LEAF, None, (), 1)
_NONE_DEF = PyTreeDef(_K_NONE, None, (), 0)


_TENSOR: type | None = None  # (core.tensor's class; that module comes later)


def is_tensor(x: Any) -> bool:
    global _TENSOR
    if _TENSOR is None:
        from .tensor import Tensor
        _TENSOR = Tensor
    return isinstance(x, _TENSOR)


def _flatten_into(node, leaves: list, is_leaf) -> PyTreeDef:
    if is_leaf is not None and is_leaf(node):
        leaves.append(node)
        return _LEAF_DEF
    if node is None:
        return _NONE_DEF
    t = type(node)
    if t in _REGISTRY:
        children, aux = _REGISTRY[t][0](node)
    elif t is list or t is tuple:
        children, aux = node, None
    elif isinstance(node, tuple) and hasattr(node, "_fields"):  # namedtuple
        children, aux = node, None
    elif t is dict:
        aux = tuple(sorted(node, key=repr))
        children = [node[k] for k in aux]
    else:
        leaves.append(node)
        return _LEAF_DEF
    n = len(leaves)
    defs = tuple([_flatten_into(c, leaves, is_leaf) for c in children])
    return PyTreeDef(t, aux, defs, len(leaves) - n)


def tree_flatten(tree: Any, is_leaf: Callable[[Any], bool] | None = None):
    leaves: list[Any] = []
    return leaves, _flatten_into(tree, leaves, is_leaf)


def _unflatten_from(d: PyTreeDef, it) -> Any:
    kind = d.kind
    if kind is _K_LEAF:
        return next(it)
    if kind is _K_NONE:
        return None
    kids = [_unflatten_from(c, it) for c in d.children]
    if kind is list:
        return kids
    if kind is tuple:
        return tuple(kids)
    if kind is dict:
        return dict(zip(d.aux, kids))
    if kind in _REGISTRY:
        return _REGISTRY[kind][1](d.aux, kids)
    return kind(*kids)  # namedtuple


def tree_unflatten(treedef: PyTreeDef, leaves) -> Any:
    return _unflatten_from(treedef, iter(leaves))


def tree_leaves(tree: Any, is_leaf=None) -> list:
    return tree_flatten(tree, is_leaf)[0]


def tree_structure(tree: Any, is_leaf=None) -> PyTreeDef:
    return tree_flatten(tree, is_leaf)[1]


def tree_map(fn: Callable, tree: Any, *rest: Any, is_leaf=None) -> Any:
    leaves, treedef = tree_flatten(tree, is_leaf)
    others = [tree_flatten(r, is_leaf)[0] for r in rest]
    return tree_unflatten(treedef, [fn(*xs) for xs in zip(leaves, *others)])


def tensor_leaves(tree: Any) -> list:
    return [x for x in tree_leaves(tree) if is_tensor(x)]
