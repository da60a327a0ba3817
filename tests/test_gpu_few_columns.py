"""Q4_0 / Q8_0 products of a few activation columns at the edges of their workgroup forms (rows and
columns that end inside a tile, K that ends inside a phase, tiles on either side of each choice), dense
and routed, against the oracle: the same floats."""
import numpy as np
import pytest

from gl import cpu_backend, gl, moe_ffn_graph, quantize, rel_err, run_on

pytestmark = pytest.mark.gpu

TYPES = [gl.Q4_0, gl.Q8_0]


@pytest.fixture(scope="module")
def hip():
    b = gl.hip_backend(0)
    yield b
    gl.libs()["core"].ggml_backend_free(b)


@pytest.fixture(scope="module")
def cpu():
    b = cpu_backend(16)
    yield b
    gl.libs()["core"].ggml_backend_free(b)


def qweight(qtype, K, N, seed, std=0.05):
    return quantize((np.random.default_rng(seed).standard_normal((N, K)) * std).astype(np.float32), qtype, impl="product")


def same(hip, cpu, build):
    a, b = run_on(hip, build), run_on(cpu, build)
    for u, v in zip(a if isinstance(a, list) else [a], b if isinstance(b, list) else [b]):
        assert np.array_equal(u, v), rel_err(u, v)


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("K,N,ncols", [
    (128, 5, 4),         # one group of four blocks, one row tile partly
    (128, 300, 63),
    (640, 37, 17),       # two phases, the second of one wave; a column tile of one column
    (3072, 200, 5),
    (13824, 64, 4),      # a row too long for the vector kernel's LDS
    (256, 8192, 16),     # 512 tiles: K split over the waves
    (256, 8200, 16),     # 513: one wave per tile
    (384, 10752, 32),    # 1344 tiles
    (384, 10768, 32),    # 1346: the GEMM
    (384, 12272, 32),
    (384, 12288, 32),
    (160, 70, 9),        # not whole groups of four blocks
])
def test_few_columns(hip, cpu, qtype, K, N, ncols):
    x = np.random.default_rng(K + ncols).standard_normal((ncols, K)).astype(np.float32)
    res = np.random.default_rng(N).standard_normal((ncols, N)).astype(np.float32)
    w = qweight(qtype, K, N, 5)

    def build(g):
        y = g.mul_mat(g.tensor(qtype, K, N, data=w), g.tensor(gl.F32, K, ncols, data=x))
        return g.add(y, g.tensor(gl.F32, N, ncols, data=res))

    same(hip, cpu, build)


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("K,N,ncols", [(256, 1000, 6), (256, 4128, 20), (640, 88, 33)])
def test_few_columns_gate_and_up(hip, cpu, qtype, K, N, ncols):
    """The SwiGLU form of both kernels, and three products of one input in one launch."""
    x = np.random.default_rng(K + ncols).standard_normal((ncols, K)).astype(np.float32)
    wg, wu, wo = qweight(qtype, K, N, 6), qweight(qtype, K, N, 7), qweight(qtype, K, 24, 8)

    def build(g):
        xt = g.tensor(gl.F32, K, ncols, data=x)
        gate = g.mul_mat(g.tensor(qtype, K, N, data=wg), xt)
        up = g.mul_mat(g.tensor(qtype, K, N, data=wu), xt)
        return [g.mul(g.silu(gate), up), g.mul_mat(g.tensor(qtype, K, 24, data=wo), xt)]

    same(hip, cpu, build)


@pytest.mark.parametrize("qtype", TYPES)
def test_few_columns_extreme_scales(hip, cpu, qtype):
    """Block scales at the ends of the F16 range: the power of two that Q4_0's dots carry is exact."""
    K, N, ncols = 512, 48, 7
    r = np.random.default_rng(11)
    w = (r.standard_normal((N, K)) * np.exp2(r.integers(-20, 12, (N, K // 32))).repeat(32, axis=1)).astype(np.float32)
    x = (r.standard_normal((ncols, K)) * np.exp2(r.integers(-16, 12, (ncols, K // 32))).repeat(32, axis=1)).astype(np.float32)
    wq = quantize(w, qtype, impl="product")
    same(hip, cpu, lambda g: g.mul_mat(g.tensor(qtype, K, N, data=wq), g.tensor(gl.F32, K, ncols, data=x)))


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n_tok", [2, 19, 70])
def test_few_columns_routed(hip, cpu, qtype, n_tok):
    r = np.random.default_rng(n_tok)
    n_embd, ff, E, k = 256, 384, 6, 2
    y = r.standard_normal((n_tok, n_embd)).astype(np.float32)
    res = r.standard_normal((n_tok, n_embd)).astype(np.float32)
    router = (r.standard_normal((E, n_embd)) * 0.1).astype(np.float32)
    wg, wu, wd = qweight(qtype, n_embd, E * ff, 1), qweight(qtype, n_embd, E * ff, 2), qweight(qtype, ff, E * n_embd, 3)

    def build(g):
        return moe_ffn_graph(g, g.tensor(gl.F32, n_embd, n_tok, data=y), g.tensor(gl.F32, n_embd, E, data=router),
                             g.tensor(qtype, n_embd, ff, E, data=wg), g.tensor(qtype, n_embd, ff, E, data=wu),
                             g.tensor(qtype, ff, n_embd, E, data=wd), k, g.tensor(gl.F32, n_embd, n_tok, data=res))

    same(hip, cpu, build)


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("first", [1, 2, 4])
@pytest.mark.parametrize("K,N,ncols", [
    (384, 100, 9),
    (640, 4100, 16),     # a 16 x 16 tile per wave
    (256, 12288, 20),    # the GEMM
    (13824, 40, 5),      # too long for the vector kernel's LDS: one column at a time unless aligned
])
def test_few_columns_weight_view(hip, cpu, qtype, first, K, N, ncols):
    """Rows that begin at any block of a larger tensor, so that their scales are aligned to 2 bytes."""
    r = np.random.default_rng(N + first)
    blocks = quantize((r.standard_normal((1, K * N + 5 * 32)) * 0.05).astype(np.float32), qtype, impl="product")
    x = r.standard_normal((ncols, K)).astype(np.float32)
    row = K // 32 * {gl.Q4_0: 18, gl.Q8_0: 34}[qtype]

    def build(g):
        w = g.view_2d(g.tensor(qtype, K * N + 5 * 32, data=blocks), K, N, row, first * (row // (K // 32)))
        return g.mul_mat(w, g.tensor(gl.F32, K, ncols, data=x))

    same(hip, cpu, build)
