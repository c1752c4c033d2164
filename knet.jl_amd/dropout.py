"""``dropout(x, p)`` and ``dropback`` (src/ops20/dropout.jl:15-42, src/ops20_gpu/dropout.jl:7-23).

The reference fills ``y`` with uniforms from the device generator (``rand!(y)``, after ``CUDA.seed!(seed)`` for a
non-zero ``seed``) and calls ``dropout_S`` in place; CPU and GPU draw from different streams, which is why its own test
only compares them statistically (test/dropout.jl:8-17).  Here the uniforms come from the library's generator in the same
way, drawn inside the dropout launch (``dropout_rand_S``: the bits of ``rand_S`` followed by ``dropout_S``); a buffer of them
can also be passed explicitly (``uniform=``) so that the device result can be compared element by element with the CPU path.
"""
import numpy as np

from . import autograd
from .activation import ActBack
from .autograd import give, primitive, recording
from .binary import AddBack
from .karray import KnetArray, number
from .libknet8 import knet8
from .random import _check, seed_


def dropout_(p, x, y):
    """``dropout!(p, x, y)``: ``y`` holds U[0,1) on entry and the result on return (in place)."""
    knet8("dropout_%s" % x.suffix, y.length, number(x, p), x.ptr, y.ptr)
    return y


def dropback_(p, x, y, dy, dx):
    """``dropback!(p, x, y, dy, dx)``."""
    knet8("dropback_%s" % x.suffix, dx.length, number(x, p), x.ptr, y.ptr, dy.ptr, dx.ptr)
    return dx


def dropback(dy, y, x, p):
    if 0 < p < 1:
        return dropback_(p, x, y, dy, x.similar())
    if p == 0:
        return dy
    if p == 1:
        from .binary import zero
        return zero(x)
    raise ValueError("Dropout probability not in [0:1]: %r" % (p,))


class DropBack:
    """``dropback(dy, y, x, p)``; no gradient for ``p``."""
    __slots__ = ("x", "y", "p")
    ends_layer = True

    def __init__(self, x, y, p):
        self.x, self.y, self.p = x, y, p

    def __call__(self, dy):
        return dropback(dy, self.y, self.x, self.p), None


@primitive
def _dropout(x, p, uniform=None, seed=0, rng=None):
    if uniform is None:
        y = x.similar()
        _check(y)
        if rng is not None:
            # position on the device: safe to capture into a graph
            knet8("dropout_rand_state_%s" % x.suffix, y.length, number(x, p), rng.ptr, x.ptr, y.ptr)
        else:
            if seed != 0:
                seed_(seed)   # if seed !== 0; CUDA.seed!(seed); end   (src/ops20_gpu/dropout.jl:13)
            knet8("dropout_rand_%s" % x.suffix, y.length, number(x, p), x.ptr, y.ptr)
        return y, DropBack(x, y, p)
    if not isinstance(uniform, KnetArray):
        uniform = KnetArray(np.asarray(uniform, dtype=x.dtype))
    else:
        uniform = uniform.copy()
    y = dropout_(p, x, uniform)
    return y, DropBack(x, y, p)


def dropout(x, p, seed=0, drop=None, uniform=None, rng=None):
    """``dropout(x, p; seed, drop)``: identity unless recording (or ``drop=True``), as in the reference.  ``uniform`` passes the
    mask buffer explicitly; ``rng`` (an ``RngState``) draws it from a generator position kept on the device."""
    from .autograd import value
    if drop is None:
        drop = recording()
    if not drop:
        return x
    if 0 < p < 1:
        return _dropout(x, p, uniform=uniform, seed=seed, rng=rng)
    if p == 0:
        return x
    if p == 1:
        from .binary import zero
        return zero(value(x))
    raise ValueError("Dropout probability not in [0:1]: %r" % (p,))


# ---- a layer's end on the tape ----------------------------------------------------------------------------------------

def _below(nodes, i, kind):
    """Position of the node that ``nodes[i]`` rests on if it was recorded right before it (leaves aside), has no gradient yet -- so ``nodes[i]`` alone uses it: later
    users have been here already -- and is of this kind; else -1."""
    node, i = nodes[i].parents[0], i - 1
    while i >= 0 and nodes[i].param is not None:
        i -= 1
    return i if i >= 0 and nodes[i] is node and node.outgrad is None and type(node.back) is kind else -1


def _layer_back(nodes, i):
    """The gradients of ``f.(z .+ b)`` and of ``dropout(relu.(z .+ b))`` as a program writes them, for z and the bias b in one launch (``Fback_biasgrad_S``, with dropout
    ``dropreluback_biasgrad_S``) instead of two or three: of an (m,n) layer dy and y are read and dz is written, where the separate launches read and write five arrays,
    with dropout eight.  (4096,2048) fp32, arrays not in cache, 26 us -> 18, with dropout 45 -> 18; (64,100) 7.3 -> 4.3 us, 11.6 -> 4.5.  dz has the same bits either way;
    every node gets the gradients that the rules one by one would give it, in the same order."""
    top, dy, p, act = i, nodes[i].outgrad, None, None
    if not isinstance(dy, KnetArray):
        return False
    y, back = nodes[i].value, nodes[i].back
    if type(back) is DropBack:
        p = back.p
        i = _below(nodes, i, ActBack)
        if i < 0 or nodes[i].back.name != "reluback":
            return False
        back = nodes[i].back
    if type(back) is ActBack:
        act = back.name
        i = _below(nodes, i, AddBack)
        if i < 0:
            return False
        back = nodes[i].back
    b, (zn, bn) = back.y, nodes[i].parents
    dims, S = dy.dims, dy.suffix
    if zn is None or bn is None or not isinstance(b, KnetArray) or b.dtype != dy.dtype or S is None or len(dims) != 2:
        return False
    m, n = dims
    if b.dims != (m, 1) or m < 2 or n < 2 or m * n >= 1 << 31 or not isinstance(back.x, KnetArray) or back.x.dims != dims or y.dims != dims or y.dtype != dy.dtype:
        return False
    dz, db = dy.similar(), b.similar()
    if p is None:
        knet8("%s_biasgrad_%s" % (act, S), m, n, dy.ptr, y.ptr, dz.ptr, db.ptr)
    else:
        knet8("dropreluback_biasgrad_%s" % S, m, n, number(dy, p), dy.ptr, y.ptr, dz.ptr, db.ptr)
    give(zn, dz)
    give(bn, db)
    for node in nodes[i:top + 1]:
        if node.param is None:
            node.outgrad = node.back = node.value = None
    return True


autograd.layer_back = _layer_back
