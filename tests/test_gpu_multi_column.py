"""Products of several activation columns at the edges of their workgroup shapes (rows and columns
that end inside a tile, one super-block, several chunks), dense and routed, against the oracle: the
same floats (every kernel adds the oracle's terms in the oracle's order)."""
import ctypes as C

import numpy as np
import pytest

from gl import Graph, attention_graph, cpu_backend, gl, moe_ffn_graph, quantize, rel_err, run_on
from test_gpu_ops import profiled

pytestmark = pytest.mark.gpu


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


def rng(seed):
    return np.random.default_rng(seed)


def qweight(qtype, K, N, seed, std=0.02):
    return quantize((rng(seed).standard_normal((N, K)) * std).astype(np.float32), qtype, impl="product")


KQUANTS = [gl.Q4_K, gl.Q5_K, gl.Q6_K]


@pytest.mark.parametrize("qtype", KQUANTS)
@pytest.mark.parametrize("K,N,ncols", [
    (256, 16420, 17),    # a 64-row workgroup per CU, the second column tile with one column
    (256, 9000, 2),      # one-wave workgroups
    (4352, 100, 33),     # K over eight waves: three chunks, the last with one super-block
    (256, 8190, 16),     # 128 tiles of 64 x 16: K over the waves
    (256, 2700, 40),     # 129
    (8192, 2690, 33),    # 129 and long rows: K over the waves for Q6_K
    (512, 4112, 250),    # 64 x 48 tiles, rows and columns ending inside one
    (768, 530, 65),      # 32 x 64 tiles
])
def test_kquant_columns(hip, cpu, qtype, K, N, ncols):
    w = qweight(qtype, K, N, K + N)
    x = rng(ncols).standard_normal((ncols, K)).astype(np.float32)
    x[0] = 0.0                      # a column of zero super-blocks
    x[1, :256] = 1.5                # one whose values are all the largest
    x[1, ::3] *= -1.0

    def build(g):
        return g.mul_mat(g.tensor(qtype, K, N, data=w), g.tensor(gl.F32, K, ncols, data=x))

    a, b = run_on(hip, build), run_on(cpu, build)
    assert np.array_equal(a, b), rel_err(a, b)


@pytest.mark.parametrize("qtype", KQUANTS)
@pytest.mark.parametrize("n_embd,ff,E,k,n_tok", [
    (512, 256, 8, 4, 130),     # items of up to 32 columns
    (2304, 256, 16, 4, 40),    # items of 16 columns whose K does not fit the LDS at once
    (512, 512, 16, 2, 33),     # items of 8
    (256, 256, 64, 8, 4),      # items of 2, most experts without a column
])
def test_kquant_expert_columns(hip, cpu, qtype, n_embd, ff, E, k, n_tok):
    r = rng(n_embd + n_tok)
    y, res = (r.standard_normal((n_tok, n_embd)).astype(np.float32) for _ in range(2))
    router = (r.standard_normal((E, n_embd)) * 0.05).astype(np.float32)
    wg, wu = (qweight(qtype, n_embd, E * ff, s, std=0.05) for s in (71, 72))
    wd = qweight(qtype, ff, E * n_embd, 73, std=0.05)

    def build(g):
        return moe_ffn_graph(g, g.tensor(gl.F32, n_embd, n_tok, data=y), g.tensor(gl.F32, n_embd, E, data=router),
                             g.tensor(qtype, n_embd, ff, E, data=wg), g.tensor(qtype, n_embd, ff, E, data=wu),
                             g.tensor(qtype, ff, n_embd, E, data=wd), k, g.tensor(gl.F32, n_embd, n_tok, data=res))

    a, b = run_on(hip, build), run_on(cpu, build)
    assert np.array_equal(a, b), rel_err(a, b)


def test_kquant_expert_columns_past_4_gib(hip, cpu):
    """Routed columns whose quantized form passes 4 GiB (columns * K above 1.9e9): the last tokens are
    read past that offset."""
    K, N, E, T, R, last = 32768, 64, 2, 58300, 200, 60      # 2.25 bytes a value: 2**32 is at token 58256
    r = rng(31)
    rows = r.standard_normal((R, K)).astype(np.float32)
    pick = r.integers(0, R, T).astype(np.int32)              # token t is row pick[t]
    ids = r.integers(0, E, (T, 1)).astype(np.int32)
    w = qweight(gl.Q4_K, K, E * N, 32)

    def build(g, pick, ids):
        x = g.get_rows(g.tensor(gl.F32, K, R, data=rows), g.tensor(gl.I32, len(pick), data=pick))
        x = g.reshape_3d(x, K, 1, len(pick))
        return g.mul_mat_id(g.tensor(gl.Q4_K, K, N, E, data=w), x, g.tensor(gl.I32, 1, len(ids), data=ids))

    a = run_on(hip, lambda g: build(g, pick, ids)).reshape(T, N)
    b = run_on(cpu, lambda g: build(g, pick[-last:], ids[-last:])).reshape(last, N)
    assert np.array_equal(a[-last:], b), rel_err(a[-last:], b)


@pytest.mark.parametrize("qtype", [gl.Q5_K, gl.Q6_K])
def test_kquant_many_experts(hip, cpu, qtype):
    """More experts than the expert lists hold: each column reads its own."""
    K, N, E, k, T = 256, 8, 4100, 2, 3
    r = rng(41)
    x, x2 = (r.standard_normal((T, n, K)).astype(np.float32) for n in (1, k))
    ids = r.integers(0, E, (T, k)).astype(np.int32)
    ids[0] = (0, E - 1)
    w = qweight(qtype, K, E * N, 42)

    def build(g):
        wt, it = g.tensor(qtype, K, N, E, data=w), g.tensor(gl.I32, k, T, data=ids)
        return [g.mul_mat_id(wt, g.tensor(gl.F32, K, v.shape[1], T, data=v), it) for v in (x, x2)]

    for a, b in zip(run_on(hip, build), run_on(cpu, build)):
        assert np.array_equal(a, b), rel_err(a, b)


def run_with_weights_at_8_bytes(backend, qtype, K, N, w, build):
    """build(g, wt) with the weights 8 bytes past the alignment of a buffer of their own."""
    core = gl.libs()["core"]
    for name in ("ggml_backend_get_default_buffer_type", "ggml_backend_buft_alloc_buffer", "ggml_backend_buffer_get_base"):
        getattr(core, name).restype = C.c_void_p
    core.ggml_backend_get_default_buffer_type.argtypes = [C.c_void_p]
    core.ggml_backend_buft_alloc_buffer.argtypes = [C.c_void_p, C.c_size_t]
    core.ggml_backend_buffer_get_base.argtypes = [C.c_void_p]
    core.ggml_backend_tensor_alloc.argtypes = [C.c_void_p, gl.T, C.c_void_p]
    buf = C.c_void_p(core.ggml_backend_buft_alloc_buffer(core.ggml_backend_get_default_buffer_type(backend), w.nbytes + 1024))
    with Graph() as g:
        wt = g.tensor(qtype, K, N, data=w)
        core.ggml_backend_tensor_alloc(buf, wt, core.ggml_backend_buffer_get_base(buf) + 8)
        out = g.compute(backend, build(g, wt))
    core.ggml_backend_buffer_free(buf)
    return out


@pytest.mark.parametrize("qtype", [gl.Q4_K, gl.Q5_K])
@pytest.mark.parametrize("ncols", [5, 70])
def test_kquant_weights_at_8_bytes(hip, cpu, qtype, ncols):
    """Weights that a caller placed 8 bytes past the buffer's alignment."""
    K, N = 512, 100
    w = qweight(qtype, K, N, 51)
    x = rng(52).standard_normal((ncols, K)).astype(np.float32)
    a, b = (run_with_weights_at_8_bytes(v, qtype, K, N, w, lambda g, wt: g.mul_mat(wt, g.tensor(gl.F32, K, ncols, data=x)))
            for v in (hip, cpu))
    assert np.array_equal(a, b), rel_err(a, b)


def test_attention_before_weights_at_8_bytes(hip, cpu):
    """The same of an O projection: the attention of 70 queries, in groups of 64, writes the one-column form."""
    hd, n_head, n_head_kv, n_kv, n_new = 128, 24, 8, 2300, 70
    r = rng(53)
    kc, vc = (r.standard_normal((n_kv, n_head_kv, hd)).astype(np.float16) for _ in range(2))
    q = r.standard_normal((n_new, n_head, hd)).astype(np.float32)
    mask = np.triu(np.full((n_new, n_kv), -np.inf, dtype=np.float32), n_kv - n_new + 1)
    K, N = n_head * hd, 64
    w = qweight(gl.Q4_K, K, N, 54)
    a, b = (run_with_weights_at_8_bytes(v, gl.Q4_K, K, N, w, lambda g, wt: g.mul_mat(
        wt, attention_graph(g, hd, n_head, n_head_kv, n_kv, n_new, n_kv, kc, vc, q, mask))) for v in (hip, cpu))
    assert np.array_equal(a, b), rel_err(a, b)


@pytest.mark.parametrize("third", [False, True])
@pytest.mark.parametrize("gtype,utype", [(gl.Q4_K, gl.Q6_K), (gl.Q6_K, gl.Q5_K), (gl.Q4_0, gl.Q4_K)])
def test_swiglu_of_two_types(hip, cpu, gtype, utype, third):
    """Gate and up of different types over a prompt: silu, product and quantization in one launch, unless
    up's launch would write a third product before the silu's turn."""
    K, F, T = 256, 512, 70
    x = rng(61).standard_normal((T, K)).astype(np.float32)
    wg, wu, wd, w3 = qweight(gtype, K, F, 62), qweight(utype, K, F, 63), qweight(gl.Q4_K, F, K, 64), qweight(utype, K, 32, 65)

    def build(g):
        xt = g.tensor(gl.F32, K, T, data=x)
        silu = g.silu(g.mul_mat(g.tensor(gtype, K, F, data=wg), xt))
        act = g.mul(silu, g.mul_mat(g.tensor(utype, K, F, data=wu), xt))
        outs = [g.mul_mat(g.tensor(gl.Q4_K, F, K, data=wd), act)]
        return outs + [g.mul_mat(g.tensor(utype, K, 32, data=w3), xt)] if third else outs

    a, names = profiled(hip, lambda: run_on(hip, build))
    b = run_on(cpu, build)
    assert ("swiglu" in names) != third, names
    for u, v in zip(a if third else [a], b if third else [b]):
        assert np.array_equal(u, v), rel_err(u, v)


@pytest.mark.parametrize("n_tok", [5, 70])
def test_kquant_activations_share_buffers(hip, cpu, n_tok):
    """Activations of one size, whose quantized forms take each other's buffers once their readers are
    launched. A SwiGLU's and a norm's, which exist in no other form, are read again by another type after
    others came and went; one is read again through a reshape, one is an output."""
    K, T = 512, n_tok
    x = rng(81).standard_normal((T, K)).astype(np.float32)
    s = (1 + 0.1 * rng(82).standard_normal(K)).astype(np.float32)
    types = {"gate": gl.Q4_K, "up": gl.Q4_K, "a4": gl.Q4_K, "a6": gl.Q6_K, "p": gl.Q5_K, "n4": gl.Q4_K, "n5": gl.Q5_K,
             "b4": gl.Q4_K, "b6": gl.Q6_K, "c": gl.Q6_K}
    w = {k: qweight(t, K, K, 83 + i, std=0.05) for i, (k, t) in enumerate(types.items())}

    def build(g):
        st, xt = g.tensor(gl.F32, K, data=s), g.tensor(gl.F32, K, T, data=x)
        wt = {k: g.tensor(t, K, K, data=w[k]) for k, t in types.items()}
        a = g.mul(g.silu(g.mul_mat(wt["gate"], xt)), g.mul_mat(wt["up"], xt))
        p = g.mul_mat(wt["a4"], a)
        q = g.mul_mat(wt["p"], p)                              # p is done with
        n = g.mul(g.rms_norm(q, 1e-5), st)
        b = g.mul(g.mul_mat(wt["n4"], n), st)
        r = g.mul_mat(wt["b4"], b)
        c = g.mul(r, st)
        out = [c, g.mul_mat(wt["c"], c), g.mul_mat(wt["a6"], a), g.mul_mat(wt["n5"], n)]
        return out + [g.mul_mat(wt["b6"], g.reshape_2d(b, K, T)), g.mul_mat(wt["c"], g.mul(out[1], st)), g.mul_mat(wt["p"], c)]

    for u, v in zip(run_on(hip, build), run_on(cpu, build)):
        assert np.array_equal(u, v), rel_err(u, v)
