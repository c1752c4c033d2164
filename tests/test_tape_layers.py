"""The gradients of a layer's end -- activation, bias, dropout -- in one launch: which tapes it takes (on the CPU, with a recorder in the place of the library) and that
every gradient is the one of the rules one by one."""
import sys

import numpy as np
import pytest

from test_host_dispatch import rec  # noqa: F401  (the recorder and its arrays)


@pytest.fixture
def tape(knet, rec, monkeypatch):  # noqa: F811
    monkeypatch.setattr(knet.libknet8(), "call", lambda fun, *a: 0)
    return rec


def one_by_one(knet, monkeypatch):
    monkeypatch.setattr(sys.modules["knet_jl_amd.autograd"], "layer_back", lambda nodes, i: False)


def launches(knet, calls, f):
    n0 = len(calls)
    J = knet.diff(f)
    return J, [c[0] for c in calls[n0:]]


@pytest.mark.parametrize("act", ["relu", "sigm", "tanh", "elu", "selu"])
def test_activation_and_bias_take_one_launch(knet, tape, act):
    calls, arr = tape
    z, b = knet.Param(arr((64, 100))), knet.Param(arr((64, 1)))
    J, names = launches(knet, calls, lambda: knet.sum(knet.mul(getattr(knet, act)(knet.add(z, b)), arr((64, 100)))))
    assert "%sback_biasgrad_32" % act in names and "%sback_32_11" % act not in names and names.count("sum_32_21") == 0
    assert knet.grad(J, z).dims == (64, 100) and knet.grad(J, b).dims == (64, 1)


def test_dropout_joins_relu_only(knet, tape):
    calls, arr = tape
    z, b, c = knet.Param(arr((64, 100), np.float64)), knet.Param(arr((64, 1), np.float64)), arr((64, 100), np.float64)
    _, names = launches(knet, calls, lambda: knet.sum(knet.mul(knet.dropout(knet.relu(z + b), 0.5), c)))
    assert "dropreluback_biasgrad_64" in names and "dropback_64" not in names
    _, names = launches(knet, calls, lambda: knet.sum(knet.mul(knet.dropout(knet.tanh(z + b), 0.5), c)))
    assert "dropback_64" in names and "tanhback_biasgrad_64" in names       # the activation and the bias still go together
    _, names = launches(knet, calls, lambda: knet.sum(knet.mul(knet.dropout(z + b, 0.5), c)))
    assert "dropback_64" in names and not any("biasgrad" in x for x in names)


def test_other_tapes_go_rule_by_rule(knet, tape):
    calls, arr = tape
    P = knet.Param
    z, b, c = P(arr((64, 100))), P(arr((64, 1))), arr((64, 100))

    def used_twice():
        h = knet.relu(z + b)
        return knet.sum(knet.mul(knet.dropout(h, 0.5), c)) + knet.sum(knet.mul(h, c))

    def sum_used_twice():
        s = z + b
        return knet.sum(knet.mul(knet.relu(s), c)) + knet.sum(knet.mul(s, c))

    def apart():
        s = z + b
        t = knet.mul(z, c)
        return knet.sum(knet.mul(knet.relu(s), t))
    tapes = [sum_used_twice, apart] + [lambda x=x, y=y: knet.sum(knet.relu(x + y)) if x.value.length == 1 else knet.sum(knet.mul(knet.relu(x + y), c if (x.value.dims == (64, 100)) else x.value))
                                       for x, y in ((z, P(arr((1, 100)))), (z, P(arr((64, 100)))), (P(arr((1, 100))), P(arr((1, 1)))), (P(arr((64, 1))), P(arr((64, 1)))))]
    tapes += [lambda: knet.sum(knet.mul(knet.relu(z + arr((64, 1))), c)), lambda: knet.sum(knet.mul(knet.relu(arr((64, 100)) + b), c)), lambda: knet.sum(knet.mul(knet.relu(b + z), c)),
              lambda: knet.sum(knet.mul(knet.relu(z + 1.0), c)), lambda: knet.sum(knet.mul(knet.gelu(z + b), c))]
    for f in tapes:
        assert not any("biasgrad" in x for x in launches(knet, calls, f)[1])
    _, names = launches(knet, calls, used_twice)     # dropout by itself; relu and the bias with the sum of both gradients
    assert "dropback_32" in names and "reluback_biasgrad_32" in names and "dropreluback_biasgrad_32" not in names


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m,n", [(64, 100), (10, 100), (33, 17), (2, 2), (257, 300), (1001, 129)])
@pytest.mark.parametrize("pdrop", [0.0, 0.5])
def test_gradients_are_those_of_the_rules_one_by_one(knet, monkeypatch, dt, m, n, pdrop):
    """Whole numbers of a few digits (and halves for dropout's division): every sum is exact in either type whatever its order, so all gradients have the same bits."""
    rng = np.random.default_rng(m * 1000 + n)
    k = 5
    whole = lambda *d: rng.integers(-4, 5, size=d).astype(dt)  # noqa: E731
    w1, b1, w2, b2 = (knet.Param(knet.KnetArray(whole(*d))) for d in ((m, k), (m, 1), (3, m), (3, 1)))
    x, c, u = knet.KnetArray(whole(k, n)), knet.KnetArray(whole(3, n)), rng.random((m, n)).astype(dt)

    def loss():
        h = knet.relu(w1 @ x + b1)
        if pdrop:
            h = knet.dropout(h, pdrop, uniform=u)
        return knet.sum(knet.mul(w2 @ h + b2, c))

    def grads():
        J = knet.diff(loss)
        return [knet.Array(knet.grad(J, p)).tobytes() for p in (w1, b1, w2, b2)]
    got = grads()
    one_by_one(knet, monkeypatch)
    assert got == grads()
    knet.libknet8().check()


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["sigm", "tanh", "elu", "selu"])
def test_other_activations(knet, monkeypatch, act):
    rng = np.random.default_rng(5)
    for dt, u in ((np.float32, 2.0 ** -24), (np.float64, 2.0 ** -53)):
        z, b, c = (rng.standard_normal(d).astype(dt) for d in ((101, 77), (101, 1), (101, 77)))
        pz, pb, cd = knet.Param(knet.KnetArray(z)), knet.Param(knet.KnetArray(b)), knet.KnetArray(c)

        def grads():
            J = knet.diff(lambda: knet.sum(knet.mul(getattr(knet, act)(pz + pb), cd)))
            return knet.Array(knet.grad(J, pz)), knet.Array(knet.grad(J, pb))
        gz, gb = grads()
        with monkeypatch.context() as one:
            one_by_one(knet, one)
            hz, hb = grads()
        assert gz.tobytes() == hz.tobytes()
        # two orders of one sum of 77 terms: each within 77 u / (1 - 77 u) * sum |dz| of it
        assert (np.abs(gb - hb) <= 2 * 77 * u / (1 - 77 * u) * np.abs(gz).sum(axis=1, keepdims=True)).all()
    knet.libknet8().check()
