"""GPU parity of the strip GEMM (k_gemm_strip.hip) at the edges of its tiles,
its partial last k-tile and its split sums, against an fp64 product.

Bound per element: the product, its sum with the bias and that with the
residual are each rounded to bf16 once (at most 2^-8 of the value rounded, so
3 * 2^-8 of the magnitudes), and the fp32 sums add K * 2^-24 of the absolute
products.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rew_amd import eager as E
from rew_amd import nn
from rew_amd import ops as O
from rew_amd.eager import DType


def _bf16(r, shape, scale):
    return E.bf16_bits_to_f32(E.f32_to_bf16_bits((r.standard_normal(shape) * scale)
                                                 .astype(np.float32))).reshape(shape)


def _dev(a):
    return E.fromHost(a, DType.BFLOAT16)


# M, K, N, row blocks per tile, whether k is split
LINEAR = [
    (1, 64, 8, 1, False),          # one row, one k-tile, fewer columns than a wave
    (32, 8, 128, 1, False),        # K below a k-tile; exactly one tile
    (33, 136, 264, 1, False),      # a second row tile of one row, K and N remainders
    (64, 1000, 392, 1, False),     # partial last k-tile with 16 of them
    (161, 2048, 520, 1, True),     # split sums with a ragged last row tile
    (8, 14336, 256, 1, True),      # the deepest split
    (129, 1032, 136, 1, True),     # split, partial last k-tile in the last split only
    (161, 72, 8200, 2, False),     # every number of row blocks: ragged last row tiles,
    (33, 4104, 4104, 2, True),     # partial last k-tiles, N remainders
    (700, 72, 5128, 4, False),
    (97, 4104, 8200, 4, True),
    (130, 4104, 8200, 5, True),
]


def _plan(name):
    r, s = name.rsplit(" r", 1)[1].split(" s")
    return int(r), int(s) > 1


@pytest.mark.parametrize("M,K,N,R,split", LINEAR)
def test_strip_linear_and_residual(gpu, M, K, N, R, split):
    r = np.random.default_rng(M * 7 + K + N)
    x, w, b = _bf16(r, (M, K), 1.0), _bf16(r, (K, N), 0.05), _bf16(r, (N,), 1.0)
    res = _bf16(r, (M, N), 1.0)
    xt, wt, bt, rt = _dev(x), _dev(w), _dev(b), _dev(res)
    exact = x.astype(np.float64) @ w.astype(np.float64)
    mag = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)
    for add in (False, True):
        def fn():
            y = nn.Linear(wt, bt).forward(xt)
            return O.add(rt, y) if add else y
        E.profileBegin()
        got = E.toHostF32(fn())
        names = [n for n, _, _ in E.profileEnd()]
        assert len(names) == 1 and names[0].startswith("gemm_lds_nn_strip+bias"), names
        assert _plan(names[0]) == (R, split), names
        want = exact + b + (res if add else 0)
        size = np.abs(exact) + np.abs(b) + (np.abs(res) if add else 0)
        assert np.all(np.abs(got - want) <= 3 * 2.0 ** -8 * size + K * 2.0 ** -24 * mag)
        for _ in range(3):  # the split sums run in one order whatever finishes last
            np.testing.assert_array_equal(E.toHostF32(fn()), got)


@pytest.mark.parametrize("T,H,I,R,split", [
    (1, 64, 8, 1, False), (33, 136, 264, 1, False), (40, 2048, 384, 1, True),
    (150, 1032, 200, 1, True), (161, 72, 8200, 2, False), (33, 2056, 5128, 2, True),
    (97, 8200, 5128, 4, True), (130, 4104, 8200, 5, True),
])
def test_strip_swiglu(gpu, oracle, T, H, I, R, split):
    """The gate and up products of every number of row blocks; a down projection
    of 8 columns reads every element of theirs."""
    rb = oracle.round_bf16
    r = np.random.default_rng(T + H + I)
    x = _bf16(r, (T, H), 1.0)
    ws = [_bf16(r, s, 0.02) for s in ((H, I), (H, I), (I, 8))]
    bs = [_bf16(r, (n,), 0.5) for n in (I, I, 8)]
    ffn = nn.GatedFeedForward(*[nn.Linear(_dev(w), _dev(b)) for w, b in zip(ws, bs)])
    xt = _dev(x.reshape(1, T, H))
    E.profileBegin()
    got = E.toHostF32(ffn.forward(xt)).reshape(T, 8)
    names = [n for n, _, _ in E.profileEnd()]
    dual = [n for n in names if n.startswith("gemm_lds_swiglu_strip")]
    assert len(dual) == 1 and _plan(dual[0]) == (R, split), names
    f = lambda y, i: rb(rb((y.astype(np.float64) @ ws[i]).astype(np.float32)) + bs[i])  # noqa: E731
    gate, up = f(x, 0), f(x, 1)
    want = f(rb(gate * (np.float32(1) / (np.float32(1) + np.exp(-gate))) * up), 2)
    # two roundings to bf16 behind the sums, and roundings of the hidden row
    # that sums in another order move by one bf16 ulp now and then
    assert np.all(np.linalg.norm(got - want, axis=0) <= 4e-3 * np.linalg.norm(want, axis=0))
    for _ in range(3):
        np.testing.assert_array_equal(E.toHostF32(ffn.forward(xt)).reshape(T, 8), got)


@pytest.mark.parametrize("M,K,N", [(33, 136, 264), (161, 2048, 520), (33, 4104, 4104)])
def test_strip_views(gpu, M, K, N):
    """Rows of a wider matrix times columns of a wider weight: the bits of dense ones."""
    r = np.random.default_rng(M + K)
    x, w = _bf16(r, (M, K + 24), 1.0), _bf16(r, (K, N + 40), 0.05)
    E.profileBegin()
    got = E.toHost(O.matmul(O.slice_(_dev(x), [0, 16], [M, 16 + K]),
                            O.slice_(_dev(w), [0, 32], [K, 32 + N])))
    names = [n for n, _, _ in E.profileEnd()]
    assert any("_strip[" in n for n in names), names
    want = E.toHost(O.matmul(_dev(np.ascontiguousarray(x[:, 16:16 + K])),
                             _dev(np.ascontiguousarray(w[:, 32:32 + N]))))
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("M,K,N", [(33, 136, 264), (161, 2048, 520), (129, 1032, 136)])
def test_strip_infinities(gpu, M, K, N):
    """Infinities and NaN reach their row and column and nothing else, past the
    partial last k-tile and through the split sums."""
    r = np.random.default_rng(M + N)
    x, w = _bf16(r, (M, K), 1.0), _bf16(r, (K, N), 0.05)
    clean = E.toHostF32(O.matmul(_dev(x), _dev(w)))
    x[3, 5], x[M - 1, K - 1], w[7, 9], w[K - 1, N - 1] = np.inf, -np.inf, np.nan, np.inf
    got = E.toHostF32(O.matmul(_dev(x), _dev(w)))
    with np.errstate(invalid="ignore"):
        want = (x.astype(np.float64) @ w.astype(np.float64)).astype(np.float32)
    odd = ~np.isfinite(want)
    np.testing.assert_array_equal(got[odd], want[odd])
    np.testing.assert_array_equal(got[~odd], clean[~odd])
    assert odd.sum() == 2 * (M + N) - 4


@pytest.mark.parametrize("B,S", [(1, 1), (2, 33)])
def test_strip_projections_with_rope(gpu, oracle, B, S):
    """The q / k / v projections of a few tokens in one launch, k split."""
    H, nh, nkv, hd = 1024, 8, 2, 128
    r = np.random.default_rng(B + S)
    x = _bf16(r, (B * S, H), 1.0)
    lin = [(_bf16(r, (H, n), 0.03), _bf16(r, (n,), 0.2)) for n in (nh * hd, nkv * hd, nkv * hd)]
    rope = nn.RotaryPositionEncoding.init(hd, S, 10000.0)
    c, s = nn.rope_tables(hd, S, 10000.0)

    def fn():
        xt = _dev(x)
        outs = []
        for (w, b), n, rot in zip(lin, (nh, nkv, nkv), (True, True, False)):
            y = O.reshape(nn.Linear(_dev(w), _dev(b)).forward(xt), [B, S, n, hd])
            y = O.transpose(y, [0, 2, 1, 3])
            outs.append(rope.forward(y) if rot else O.add(y, y))
        return outs

    E.profileBegin()
    outs = [E.toHostF32(t) for t in fn()]
    names = [n for n, _, _ in E.profileEnd()]
    sets = [n for n in names if n.startswith("gemm_lds_nn_strip{") and n.count("+rope") == 2]
    assert len(sets) == 1 and _plan(sets[0]) == (1, True), names
    for got, (w, b), n, rot in zip(outs, lin, (nh, nkv, nkv), (True, True, False)):
        y = oracle.round_bf16(oracle.round_bf16((x.astype(np.float64) @ w).astype(np.float32)) + b)
        y = y.reshape(B, S, n, hd).transpose(0, 2, 1, 3)
        want = oracle.rope(np.ascontiguousarray(y), c, s, offset=0) if rot else y + y
        assert np.linalg.norm(got - want) <= 4e-3 * np.linalg.norm(want)


ROPE_CHILD = r"""
import sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from test_gpu_gemm_strip import rope_sets
from rew_amd import eager as E
E.installEagerBackend(E.mi355x(0))
np.savez(sys.argv[2], *rope_sets("gemm_lds_nn{"))
"""


def rope_sets(label):
    """q / k / v projections with ragged row and column tiles of either kernel."""
    r = np.random.default_rng(12)
    res = []
    for B, S, nh, nkv, hd, H in ((2, 33, 3, 1, 24, 136), (1, 300, 5, 2, 72, 264)):
        x = _dev(_bf16(r, (B * S, H), 1.0))
        rope = nn.RotaryPositionEncoding.init(hd, S, 10000.0)
        outs = []
        E.profileBegin()
        for n, rot in ((nh, True), (nkv, True), (nkv, False)):
            w, b = _bf16(r, (H, n * hd), 0.05), _bf16(r, (n * hd,), 0.2)
            y = O.reshape(nn.Linear(_dev(w), _dev(b)).forward(x), [B, S, n, hd])
            y = O.transpose(y, [0, 2, 1, 3])
            outs.append(rope.forward(y) if rot else O.add(y, y))
        E.flush()
        names = [n for n, _, _ in E.profileEnd()]
        assert any(n.startswith(label) and n.count("+rope") == 2 for n in names), names
        res += [E.toHostF32(t) for t in outs]
    return res


def test_rope_sets_equal_the_256_tiles(gpu, tmp_path):
    """Unsplit sets on both kernels: the same sums in the same order."""
    import os
    import subprocess
    import sys
    from pathlib import Path
    out = str(tmp_path / "sets.npz")
    p = subprocess.run([sys.executable, "-c", ROPE_CHILD,
                        str(Path(__file__).resolve().parents[1]), out],
                       env=dict(os.environ, REW_MI355X_GEMM_TILE="lds"), capture_output=True,
                       text=True, timeout=90)
    assert p.returncode == 0, p.stderr[-3000:]
    ref = np.load(out)
    for i, got in enumerate(rope_sets("gemm_lds_nn_strip{")):
        np.testing.assert_array_equal(got, ref[f"arr_{i}"])


def test_reversed_rows(gpu):
    """A view with a negative row stride takes none of the kernels that form
    unsigned offsets from the view's base."""
    def flip(t):
        return E.dispatchEager("reverse", [t], [("dimensions", "[0]")])[0]

    r = np.random.default_rng(11)
    for M, K, N in ((40, 256, 264), (2048, 64, 4096)):
        x, w = _bf16(r, (M, K), 1.0), _bf16(r, (K, N), 0.05)
        got = E.toHostF32(O.matmul(flip(_dev(x)), _dev(w)))
        want = E.toHostF32(O.matmul(_dev(np.ascontiguousarray(x[::-1])), _dev(w)))
        assert np.linalg.norm(got - want) <= 2e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("M,K,N,strip", [
    (1000, 1024, 8192, False), (600, 4096, 14336, False), (3000, 64, 4096, False),
    (4000, 256, 1408, False), (1500, 4096, 4096, False), (1400, 4096, 4096, False),
    (1200, 4096, 4096, True), (8, 1024, 128256, True), (16, 4096, 14336, True),
])
def test_strip_or_256_tiles(gpu, M, K, N, strip):
    """Which kernel takes a Linear: the strip kernel below 96 tiles of 256x256,
    and past that for few rows over many weights only."""
    w, b = E.empty(DType.BFLOAT16, (K, N)), E.empty(DType.BFLOAT16, (N,))
    E.profileBegin()
    out = nn.Linear(w, b).forward(E.empty(DType.BFLOAT16, (M, K)))
    E.flush()
    names = [n for n, _, _ in E.profileEnd()]
    del out
    assert len(names) == 1 and ("_strip" in names[0]) == strip, names


@pytest.mark.parametrize("T,H,I,strip", [
    (300, 4096, 14336, False), (600, 4096, 14336, False), (6000, 2048, 1408, False),
    (2600, 512, 2048, False), (64, 4096, 14336, True), (1500, 2048, 1408, True),
])
def test_swiglu_strip_or_256_tiles(gpu, T, H, I, strip):
    e = lambda *s: E.empty(DType.BFLOAT16, s)  # noqa: E731
    gate, up, down = (nn.Linear(e(*s), e(s[1])) for s in ((H, I), (H, I), (I, H)))
    E.profileBegin()
    out = nn.GatedFeedForward(gate, up, down).forward(e(1, T, H))
    E.flush()
    names = [n for n, _, _ in E.profileEnd()]
    del out
    assert [("_strip" in n) for n in names if "swiglu" in n] == [strip], names
