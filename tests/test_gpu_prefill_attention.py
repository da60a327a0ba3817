"""Attention of query batches at the edges of its workgroup forms: scores in registers (up to 512, 1024,
2048, 4096 positions) or in scratch (fewer workgroups than CUs, or longer rows), partial row and
position tiles, position tiles that nobody sees in the middle of a row. The chain's floats exactly."""
import numpy as np
import pytest

from gl import cpu_backend, gl, rel_err, rel_err_floor, run_on
from test_gpu_ops import TOL, attention_graph, profiled

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


def check(hip, cpu, hd, n_head, n_head_kv, n_kv, n_new, mask, flash):
    r = np.random.default_rng(n_kv + 3 * n_new + hd)
    n_ctx = n_kv + 3
    kc = r.standard_normal((n_ctx, n_head_kv, hd)).astype(np.float16)
    vc = r.standard_normal((n_ctx, n_head_kv, hd)).astype(np.float16)
    q = r.standard_normal((n_new, n_head, hd)).astype(np.float32)

    def build(g):
        return attention_graph(g, hd, n_head, n_head_kv, n_kv, n_new, n_ctx, kc, vc, q, mask, flash)

    a, names = profiled(hip, lambda: run_on(hip, build))
    b = run_on(cpu, build)
    assert "attn_prefill" in names, names
    if flash:
        assert rel_err_floor(a, b) < TOL, rel_err_floor(a, b)
    else:
        assert np.array_equal(a, b), rel_err(a, b)


def causal(n_kv, n_new):
    mask = np.zeros((n_new, n_kv), dtype=np.float32)
    for i in range(n_new):
        mask[i, n_kv - n_new + i + 1:] = -np.inf
    return mask


@pytest.mark.parametrize("flash", [False, True])
@pytest.mark.parametrize("hd,n_head,n_head_kv,n_kv,n_new", [
    (64, 8, 8, 7, 7),          # fewer positions than a tile, waves with none
    (64, 64, 64, 512, 65),     # registers, 8 tiles a wave to the last
    (64, 64, 64, 513, 65),     # 16 tiles a wave
    (96, 64, 32, 1024, 70),
    (128, 64, 64, 1025, 65),   # 32 tiles a wave, 4 waves
    (64, 64, 64, 2049, 65),    # 8 waves
    (64, 32, 32, 4096, 200),
    (128, 16, 4, 257, 33),     # scratch, fewer workgroups than CUs
    (96, 6, 2, 2240, 5),
    (64, 8, 1, 300, 6),        # eight heads of a group in a row tile
    (96, 32, 32, 4097, 97),    # scratch, a row past the registers
    (64, 32, 32, 4100, 300),   # more row tiles than workgroups
])
def test_prefill_attention_forms(hip, cpu, hd, n_head, n_head_kv, n_kv, n_new, flash):
    check(hip, cpu, hd, n_head, n_head_kv, n_kv, n_new, causal(n_kv, n_new), flash)


@pytest.mark.parametrize("flash", [False, True])
@pytest.mark.parametrize("hd,n_head,n_head_kv,n_kv,n_new", [
    (128, 8, 2, 200, 40),      # registers
    (64, 8, 8, 700, 21),       # scratch
])
def test_prefill_attention_holes_in_the_mask(hip, cpu, hd, n_head, n_head_kv, n_kv, n_new, flash):
    r = np.random.default_rng(n_kv)
    mask = causal(n_kv, n_new)
    mask[:, 30:100] = -np.inf                       # whole tiles, one partly
    mask[:, 128:160] = -np.inf
    mask[r.random(mask.shape) < 0.2] = -np.inf
    mask[:, 0] = 0.0                                # no row without a position
    mask[:, 1] = -3.5
    check(hip, cpu, hd, n_head, n_head_kv, n_kv, n_new, mask, flash)
