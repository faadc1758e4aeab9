"""The engine drop-in (miso_amd/engine/attention.{hpp,hip}) run on MI355X, built against stand-ins of
the engine's types (oracle/drop_in_capi.hip): a 300-token prefill and a decode step give the C ABI
layer's y, h and core bit for bit, and leave every scratch member as the engine's own wiring does
(src/engine/attention.hip:76-148): the normed rows, the projections, the prepared queries, core."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from conftest import to_dev, to_host
from test_layer_gpu import EPS, layer_case  # noqa: F401  (a fixture)

pytestmark = pytest.mark.gpu

N, MAX_CTX = 300, 301


@pytest.fixture
def engine(O, attn, layer_case):  # noqa: F811
    layer, _, _ = layer_case
    lib = O.drop_in()
    mats = [layer._keep[i][0] for i in range(4)]
    e = lib.drop_engine_new((ctypes.c_void_p * 4)(*(m.data_ptr() for m in mats)),
                            (ctypes.c_uint64 * 4)(*(m.numel() for m in mats)),
                            *(t.data_ptr() for t in layer._keep[4:]), MAX_CTX, N)
    assert e

    def read(name, n):
        out = np.empty(n, np.float32)
        assert lib.drop_engine_read(e, name.encode(), out.ctypes.data, n) >= n
        return out

    yield lib, e, read
    lib.drop_engine_delete(e)


def test_engine_steps_and_scratch_members(O, attn, torch_mod, layer_case, engine):  # noqa: F811
    torch = torch_mod
    layer, deq, norms = layer_case
    lib, e, read = engine
    rng = np.random.default_rng(3)
    h0 = rng.standard_normal((N + 1, 2048)).astype(np.float32)
    delta = (0.5 * rng.standard_normal((N + 1, 2048))).astype(np.float32)
    xs = (h0 + delta).astype(np.float64)
    normed = xs / np.sqrt((xs * xs).mean(axis=1, keepdims=True) + EPS) * norms["attn_norm"]
    d = to_dev(torch, delta.reshape(-1))
    out = []
    for who in ("engine", "layer"):
        h = to_dev(torch, h0.reshape(-1))
        y = torch.zeros((N + 1) * 2048, device="cuda")
        kc = torch.zeros(2 * MAX_CTX * 256, dtype=torch.float16, device="cuda")
        vc, ws = torch.zeros_like(kc), attn.LayerWorkspace(max_tok=N)
        for a, b in ((0, N), (N, N + 1)):
            at = slice(a * 2048, b * 2048)
            torch.cuda.synchronize()
            if who == "engine":
                assert lib.drop_engine_step(e, int(b > N), h[at].data_ptr(), d[at].data_ptr(),
                                            y[at].data_ptr(), b - a, EPS) == 0
            elif b > N:
                attn.layer_decode(layer, kc, vc, MAX_CTX, a, h[at], d[at], y[at], EPS, ws)
            else:
                attn.layer_prefill(layer, kc, vc, MAX_CTX, a, b - a, h[at], d[at], y[at], EPS, ws)
            torch.cuda.synchronize()
        out.append((to_host(h), to_host(y)))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][0], (h0 + delta).ravel())
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(read("pcore", N * 4096), to_host(ws.prefill_core).ravel())
    assert np.array_equal(read("score", 4096), to_host(ws.decode_core))
    # f32 rows of the float64 norm (2048 squares summed: 1e-6); decode's and prefill's members
    for name, first, n in (("p", 0, N), ("s", N, 1)):
        xn = read(name + "xn", n * 2048).reshape(n, 2048)
        assert np.abs(xn - normed[first:first + n]).max() <= 1e-6 * np.abs(normed).max()
        proj = read(name + "proj", n * 9216).reshape(n, 9216)[:, :8192].reshape(n, 16, 2, 256)
        ref = (xn.astype(np.float16).astype(np.float64) @ deq["q"].T).reshape(n, 16, 2, 256)
        assert np.abs(proj - ref).max() <= 1e-3 * np.abs(ref).max()
        q = proj[:, :, 0].astype(np.float64)
        q = q / np.sqrt((q * q).mean(axis=2, keepdims=True) + EPS) * norms["q_norm"]
        a = np.arange(first, first + n)[:, None, None] * norms["inv_freq"].astype(np.float64)
        lo, hi = q[..., :32].copy(), q[..., 32:64].copy()
        q[..., :32], q[..., 32:64] = lo * np.cos(a) - hi * np.sin(a), hi * np.cos(a) + lo * np.sin(a)
        got = read(name + "q", n * 4096).reshape(n, 16, 256)
        # an angle of up to 300 rounds at 2^-16 in f32
        assert np.abs(got - q).max() <= 3e-5 * np.abs(q).max()
