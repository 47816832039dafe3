"""GPU learned-band predictor: features, BF16-MFMA forward and gradients
against the FP64 numpy oracle (oracle/mlp.py)."""
import itertools

import numpy as np
import pytest

import mlp as Mo
from gproshan_amd import geodesics as P
from gproshan_amd import learned as Lr
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu


def _data(n=4096, seed=0):
    rng = np.random.default_rng(seed)
    F = rng.normal(size=(n, Lr.NFEAT)).astype(np.float32)
    t = (0.1 * np.tanh(F[:, 0]) + 0.05 * F[:, 1] ** 2).astype(np.float32)
    return F, t


def _holed(n=40, seed=9):
    xyz, f = G.height_field(n, seed)
    r, c = f[:, 0] // n, f[:, 0] % n
    keep = f[~((r >= 10) & (r < 16) & (c >= 12) & (c < 20))]
    used = np.unique(keep)
    remap = np.full(len(xyz), -1, np.int64)
    remap[used] = np.arange(len(used))
    return xyz[used], remap[keep].astype(np.uint32)


@pytest.mark.parametrize("mesh", ["hf33", "holed40", "ico3"])
def test_features_match_oracle(oracle, mesh):
    """All ten per-vertex features: on an open height field, on one with an
    internal hole (border vertices inside the mesh) and on a closed sphere."""
    if mesh == "hf33":
        (xyz, f), src = G.height_field(33, 4), [100, 700]
    elif mesh == "holed40":
        (xyz, f), src = _holed(), [5, 900]
    else:
        (xyz, f), src = G.icosphere(3, 0.01, 4), [0, 300]
    M = oracle.Mesh(xyz, f)
    C = P.che(xyz, f)
    lev = M.toplesets(src)[0]
    # mean fan edge length as the library computes it (closing entries counted twice)
    Fo, eo = Mo.features(M, xyz, src, lev, _mean_edge(M, xyz))
    Fg, eg = Lr.features(C, src)
    assert np.allclose(eg, eo, rtol=1e-6, atol=1e-7)
    assert np.allclose(Fg, Fo, rtol=1e-4, atol=1e-5), np.abs(Fg - Fo).max(axis=0)


def _mean_edge(M, xyz):
    tot, cnt = 0.0, 0
    links, tris = Mo.fan_lists(M)
    for v, tl in enumerate(tris):
        if not tl:
            continue
        fan = [tl[0][0]] + [b for _, b in tl]
        for u in fan:
            tot += np.linalg.norm(xyz[u] - xyz[v])
            cnt += 1
    return tot / cnt


def test_forward_matches_oracle():
    F, _ = _data(1000, 1)
    net = Lr.MLP(seed=5)
    p = Lr.unpack(net.params())
    pb = {k: (Mo.bf16(v) if k in ("W1", "W2") else v) for k, v in p.items()}
    X = np.zeros((len(F), Mo.KPAD))
    X[:, :Mo.NF] = Mo.bf16(F)
    yo, cache = Mo.forward(X, pb)
    yg = net.forward(F)
    # BF16 rounding of the hidden activations: ~1e-2 relative
    err = np.abs(yg - yo) / (np.abs(yo).max() + 1e-6)
    assert err.max() < 3e-2, err.max()


def test_gradient_matches_oracle():
    F, t = _data(2048, 2)
    net = Lr.MLP(seed=7)
    p = Lr.unpack(net.params())
    pb = {k: (Mo.bf16(v) if k in ("W1", "W2") else v) for k, v in p.items()}
    X = np.zeros((len(F), Mo.KPAD))
    X[:, :Mo.NF] = Mo.bf16(F)
    y, cache = Mo.forward(X, pb)
    go = Mo.backward(y, t, cache, pb)
    gg, loss = net.gradient(F, t)
    gd = Lr.unpack(gg)
    assert abs(loss - Mo.loss(y, t)) <= 3e-2 * Mo.loss(y, t) + 1e-6
    for k in ("W1", "b1", "W2", "b2", "w3", "b3"):
        a, b = gd[k].reshape(-1), go[k].reshape(-1)
        rel = np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12)
        print(f"[grad] {k} rel {rel:.3e}", flush=True)
        assert rel < 5e-2, (k, rel)


def test_training_reduces_loss():
    F, t = _data(32768, 3)
    net = Lr.MLP(seed=1)
    _, l0 = net.gradient(F, t)
    net.train(F, t, steps=300, batch=4096, lr=3e-3)
    _, l1 = net.gradient(F, t)
    print(f"[train] loss {l0:.4e} -> {l1:.4e}", flush=True)
    assert l1 < 0.2 * l0


@pytest.mark.parametrize("n,copies", [(1, 2), (1, 64), (15, 4), (16, 8), (17, 2), (31, 2), (33, 4), (127, 2), (129, 8),
                                      (500, 16), (4099, 8)])
def test_gradient_does_not_depend_on_where_a_row_sits(n, copies):
    """The mean gradient of n rows is that of the same rows repeated a power of
    two times: each row's BF16 values scale exactly, only the FP32 sums are
    taken in another order.  The repeats put every row into other tiles, waves,
    workgroups and (past 32,768 rows) passes of the gradient kernel.  At most
    ~600 FP32 additions follow one another (6e-8 each): 1e-4 of the norm leaves
    a factor of three for cancellation."""
    F, t = _data(n, 11)
    net = Lr.MLP(seed=3)
    g1, l1 = net.gradient(F, t)
    g2, l2 = net.gradient(np.tile(F, (copies, 1)), np.tile(t, copies))
    assert abs(l1 - l2) <= 1e-4 * l1
    a, b = Lr.unpack(g1), Lr.unpack(g2)
    for k in a:
        assert np.linalg.norm(a[k] - b[k]) <= 1e-4 * np.linalg.norm(a[k]) + 1e-12, k


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_gradient_adds_its_waves(seed):
    """The gradient of 128 rows, one workgroup's, is the FP32 sum of those of its
    four waves' 32 rows in some order: of each weight's value one of the sums has
    the bits (the waves' shares scale by a power of two, exactly)."""
    F, t = _data(128, seed)
    net = Lr.MLP(seed=seed)
    part = [np.float32(0.25) * net.gradient(F[q:q + 32], t[q:q + 32])[0].astype(np.float32) for q in range(0, 128, 32)]
    got = Lr.unpack(net.gradient(F, t)[0])
    part = [Lr.unpack(p) for p in part]
    for k in ("W1", "W2"):
        hit = np.zeros(got[k].shape, bool)
        for order in itertools.permutations(range(4)):
            s = np.zeros(got[k].shape, np.float32)
            for w in order:
                s = s + part[w][k].astype(np.float32)
            hit |= s == got[k]
        assert hit.all(), (k, int((~hit).sum()))
