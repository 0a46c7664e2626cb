"""GPU parity of the f32 matrix-core GEMM (gemm_f32_mfma_kernel).  Each output
is the fmaf chain over k that the generic and the 16 x 16 kernels run, so a
slice of a product, small enough for the latter, has the same bits as the
product's; the generic kernel's own bits come from a process that forces it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rew_amd import eager as E
from rew_amd import nn
from rew_amd import ops as O


def dev(a):
    return E.fromHost(np.ascontiguousarray(a, np.float32))


def run(fn):
    E.profileBegin()
    out = E.toHost(fn())
    return out, [n for n, _, _ in E.profileEnd()]


FORMS = {"nn": ((1, 0), lambda a, b: O.matmul(dev(a), dev(b))),
         "nt": ((1, 1), lambda a, b: O.dotGeneral(dev(a), dev(b.T), [], [], [1], [1])),
         "tn": ((0, 0), lambda a, b: O.dotGeneral(dev(a.T), dev(b), [], [], [0], [0])),
         "tt": ((0, 1), lambda a, b: O.dotGeneral(dev(a.T), dev(b.T), [], [], [0], [1]))}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("M,K,N", [
    (577, 100, 641),    # remainders of every tile edge; 4-byte loads along m and n
    (640, 1, 640),      # one k-step
    (640, 32, 644),     # exactly one k-tile
    (600, 33, 700),     # one past it, odd K
    (1100, 96, 8260),   # 128-row tiles (9 x 130 of them)
])
def test_chain_equals_small_kernel(gpu, oracle, form, M, K, N):
    r = np.random.default_rng(M + K + N)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = (r.standard_normal((K, N)) * 10.0 ** r.integers(-3, 3, (K, N))).astype(np.float32)
    a[3, 0], b[0, 5] = np.inf, np.nan
    _, f = FORMS[form]
    got, names = run(lambda: f(a, b))
    assert any(n.startswith("gemm_f32_mfma") for n in names), names
    for m0, n0 in ((0, 0), (M - 33, N - 65), (M // 2, N // 3)):
        ref, names = run(lambda: f(a[m0:m0 + 33], b[:, n0:n0 + 65]))
        assert any(n.startswith("gemm_f32_small") for n in names), names
        part = got[m0:m0 + 33, n0:n0 + 65]
        nan = np.isnan(ref)
        np.testing.assert_array_equal(np.isnan(part), nan)
        np.testing.assert_array_equal(part[~nan].view(np.uint32), ref[~nan].view(np.uint32))
    rows = slice(4, 40)  # away from the infinity
    want = a[rows].astype(np.float64) @ b[:, 6:].astype(np.float64)
    bound = (K + 1) * 2.0 ** -24 * (np.abs(a[rows]).astype(np.float64) @ np.abs(b[:, 6:]))
    assert np.all(np.abs(got[rows, 6:] - want) <= bound)


def test_batches_and_epilogues(gpu):
    r = np.random.default_rng(5)
    B, M, K, N = 6, 333, 65, 331
    a, b = r.standard_normal((B, M, K)), r.standard_normal((B, K, N))
    got, names = run(lambda: O.dotGeneral(dev(a), dev(b), [0], [0], [2], [1]))
    assert any(n.startswith("gemm_f32_mfma") for n in names), names
    a32, b32 = a.astype(np.float32), b.astype(np.float32)
    want = np.matmul(a32.astype(np.float64), b32.astype(np.float64))
    bound = (K + 1) * 2.0 ** -24 * np.matmul(np.abs(a32).astype(np.float64), np.abs(b32))
    assert np.all(np.abs(got - want) <= bound)
    x, w, bias, res = a32[0], b32[0], r.standard_normal(N).astype(np.float32), got[1]

    def lin():
        return nn.Linear(dev(w), dev(bias)).forward(dev(x))

    x = np.repeat(x, 4, 0)
    res = np.repeat(res, 4, 0)
    plain, _ = run(lambda: O.matmul(dev(x), dev(w)))
    for fn, ref in ((lin, plain + bias), (lambda: O.add(dev(res), lin()), res + (plain + bias)),
                    (lambda: nn.relu(lin()), np.maximum(plain + bias, 0))):
        out, names = run(fn)
        assert len(names) == 1 and names[0].startswith("gemm_f32_mfma+bias"), names
        np.testing.assert_array_equal(out, ref)


@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (2, 4, 4)])
def test_batch_past_the_grid_limit(gpu, M, K, N):
    """2^24 products: more workgroups of 256 threads than one grid dimension takes."""
    r = np.random.default_rng(K)
    B = 1 << 24
    a, b = (np.resize(r.standard_normal((4099, *s)).astype(np.float32), (B, *s))
            for s in ((M, K), (K, N)))
    got = E.toHost(O.dotGeneral(dev(a), dev(b), [0], [0], [2], [1]))
    want = E.toHost(O.dotGeneral(dev(a[:4099]), dev(b[:4099]), [0], [0], [2], [1]))
    for i in range(0, B, 4099):
        part = got[i:i + 4099]
        np.testing.assert_array_equal(part, want[:len(part)])


@pytest.mark.parametrize("B,M,K,N,kernel", [
    (1500, 1, 1, 1, "gemm_generic"), (1500, 64, 7, 1, "gemm_generic"),
    (1500, 1, 7, 64, "gemm_generic"), (1500, 3, 8, 3, "gemm_generic"),
    (1500, 2, 33, 2, "gemm_generic"), (1500, 13, 15, 13, "gemm_generic"),
    (1500, 13, 16, 13, "gemm_f32_mfma"), (1500, 13, 17, 13, "gemm_f32_mfma"),
    (1500, 8, 8, 8, "gemm_f32_mfma"), (1500, 65, 7, 3, "gemm_f32_mfma"),
    (1500, 64, 8, 64, "gemm_f32_mfma"), (1500, 13, 8, 13, "gemm_generic"),
    (300, 13, 8, 13, "gemm_f32_mfma"), (300, 7, 5, 7, "gemm_f32_mfma"),
    (300, 3, 17, 3, "gemm_f32_mfma"), (300, 2, 8, 2, "gemm_generic"),
    (300, 64, 5, 1, "gemm_generic"), (300, 1, 17, 1, "gemm_generic"),
])
def test_batches_of_small_products(gpu, B, M, K, N, kernel):
    """Which kernel takes many products of one tile each, and its sums."""
    r = np.random.default_rng(M + K + N)
    a, b = (r.standard_normal((B, *s)).astype(np.float32) for s in ((M, K), (K, N)))
    got, names = run(lambda: O.dotGeneral(dev(a), dev(b), [0], [0], [2], [1]))
    assert [n.split("[")[0] for n in names] == [kernel], names
    want = np.matmul(a.astype(np.float64), b.astype(np.float64))
    bound = (K + 1) * 2.0 ** -24 * np.matmul(np.abs(a).astype(np.float64), np.abs(b))
    assert np.all(np.abs(got - want) <= bound)


def test_loads_of_four_bytes_keep_two_waves(gpu):
    """128-row tiles whose operands come 4 bytes at a time stay within the
    registers of two waves per SIMD (one ran them half as fast again)."""
    def us(n):
        a, b = E.empty(E.DType.FLOAT32, (5000, n, n)), E.empty(E.DType.FLOAT32, (5000, n, n))
        best = 1e9
        for _ in range(5):
            E.profileBegin()
            out = O.dotGeneral(a, b, [0], [0], [2], [1])
            E.flush()
            prof = E.profileEnd()
            del out
            assert len(prof) == 1 and prof[0][0].startswith("gemm_f32_mfma"), prof
            best = min(best, prof[0][2] * 1e3)
        return best

    # (measured: 281 us against 212 for 16-byte loads; 408 with one wave)
    odd, even = us(65), us(68)
    assert odd <= 1.6 * even, (odd, even)


def test_one_row_tile_keeps_its_height(gpu):
    """Many products of at most 64 rows run 64-row tiles: about twice the rate of
    128-row ones, which hold twice the LDS and load as much again for nothing."""
    def us(M):
        a, b = E.empty(E.DType.FLOAT32, (30000, M, 8)), E.empty(E.DType.FLOAT32, (30000, 8, 32))
        best = 1e9
        for _ in range(5):
            E.profileBegin()
            out = O.dotGeneral(a, b, [0], [0], [2], [1])
            E.flush()
            prof = E.profileEnd()
            del out
            assert len(prof) == 1 and prof[0][0].startswith("gemm_f32_mfma"), prof
            best = min(best, prof[0][2] * 1e3)
        return best

    # (measured: 127 us against 313; in 128-row tiles 288)
    low, high = us(32), us(100)
    assert low <= 0.65 * high, (low, high)


@pytest.mark.parametrize("M,K,N,kernel", [
    (8, 1024, 2816, "gemm_f32_small"), (16, 1024, 4096, "gemm_f32_small"),
    (17, 1024, 4096, "gemm_f32_mfma"), (32, 512, 4096, "gemm_f32_small"),
    (33, 512, 4096, "gemm_f32_mfma"), (1, 4096, 4096, "gemm_f32_small"),
    (8, 2048, 1024, "gemm_f32_small"), (9, 2048, 1024, "gemm_f32_mfma"),
    (100, 3000, 70, "gemm_f32_small"), (100, 3000, 72, "gemm_f32_mfma"),
])
def test_few_rows(gpu, M, K, N, kernel):
    """Which kernel takes a product of few rows, and its sums."""
    r = np.random.default_rng(M + K + N)
    a, b = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    got, names = run(lambda: O.matmul(dev(a), dev(b)))
    assert [n.split("[")[0] for n in names] == [kernel], names
    want = a.astype(np.float64) @ b
    bound = (K + 1) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b))
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("K", [16, 48, 40, 32, 12])
def test_products_that_underflow(gpu, form, K):
    """Sums of denormals, and zeros whose sign is the last term's: a chain ends
    at the next multiple of 16 in every kernel, with zero terms past K."""
    _, f = FORMS[form]
    a = np.full((640, K), -1e-20, np.float32)
    b = np.full((K, 648), 1e-20, np.float32)
    b[:, ::2] = 1e-30  # (the products underflow)
    got, names = run(lambda: f(a, b))
    assert any(n.startswith("gemm_f32_mfma") for n in names), names
    ref, names = run(lambda: f(a[:33], b[:, :65]))
    assert any(n.startswith("gemm_f32_small") for n in names), names
    np.testing.assert_array_equal(got[:33, :65].view(np.uint32), ref.view(np.uint32))
    assert (ref[0, 0] == 0) and np.signbit(ref[0, 0]) == (K % 16 == 0)
    assert 0 < -ref[0, 1] < 1e-37


GENERIC_CHILD = r"""
import sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from test_gpu_gemm_f32 import FORMS, generic_cases, run
from rew_amd import eager as E
E.installEagerBackend(E.mi355x(0))
out = []
for form, a, b in generic_cases():
    got, names = run(lambda: FORMS[form][1](a, b))
    assert [n.split("[")[0] for n in names] == ["gemm_generic"], names
    out.append(got)
np.savez(sys.argv[2], *out)
"""


def generic_cases():
    r = np.random.default_rng(6)
    for M, K, N in ((577, 100, 641), (640, 48, 644), (1100, 33, 8260), (64, 200, 70), (16, 64, 16),
                    (300, 128, 32), (8, 2100, 300)):
        for form in ("nn", "tt"):
            a = r.standard_normal((M, K)).astype(np.float32)
            b = (r.standard_normal((K, N)) * 10.0 ** r.integers(-3, 3, (K, N))).astype(np.float32)
            a[:, K // 2:] *= np.float32(1e-25)
            b[:, 1::3] *= np.float32(1e-16)  # sums of denormals in between
            a[3] = 1e-30
            b[:, 0] = -1e-30                 # products that underflow
            yield form, a, b


def test_equals_the_generic_kernel(gpu, tmp_path):
    """The matrix-core, 16 x 16, 8 x 8 and narrow kernels against the generic one."""
    import os
    import subprocess
    import sys
    from pathlib import Path
    out = str(tmp_path / "generic.npz")
    p = subprocess.run([sys.executable, "-c", GENERIC_CHILD,
                        str(Path(__file__).resolve().parents[1]), out],
                       env=dict(os.environ, REW_MI355X_GEMM_TILE="generic"),
                       capture_output=True, text=True, timeout=90)
    assert p.returncode == 0, p.stderr[-3000:]
    ref = np.load(out)
    seen = set()
    for i, (form, a, b) in enumerate(generic_cases()):
        got, names = run(lambda: FORMS[form][1](a, b))
        seen |= {n.split("[")[0] for n in names}
        np.testing.assert_array_equal(got.view(np.uint32), ref[f"arr_{i}"].view(np.uint32))
    assert seen == {"gemm_f32_mfma", "gemm_f32_small", "gemm_f32_narrow"}, seen
