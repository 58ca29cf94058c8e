"""Kernels over rows of the listed-layers decoders at the sizes where their vector forms begin and end."""
import ctypes as C

import numpy as np
import pytest

import plain_hybrid as ph
from gpu_calls import Gpu, View, Z, close, get, p, rand, view

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 64, 68, 1024, 1028, 2048, 2052, 4096, 4100, 1026])
@pytest.mark.parametrize("top", [1, 3, 4, 5, 9])
@pytest.mark.parametrize("second", [False, True])
def test_routed_rows_join_the_residual(hip, n, top, second):
    """The weighted sum of routed rows, normed and added: counts around the four rows on their way at a time, places without a row, rows beyond y."""
    gpu, m, rows, eps = Gpu(hip), 5, 7, 1e-3
    x, y, w, nxt, weights = rand(1, m, n), rand(2, rows, n), rand(3, n), rand(4, n), rand(5, m, top)
    slots = np.random.default_rng(6).integers(-1, rows + 1, (m, top)).astype(np.int32)
    slots[0], slots[1] = 0, -1
    y[rows - 1] = np.where(np.arange(n) % 2, 50.0, -50.0)
    want = np.zeros((m, n))
    for i in range(m):
        for j in range(top):
            if 0 <= slots[i, j] < rows:
                want[i] += weights[i, j] * y[slots[i, j]]
    want = x + ph.rms(want, eps) * w
    sx, sy, sw, sn, ss, swt = gpu.up(x), gpu.up(y), gpu.up(w), gpu.up(nxt), gpu.up(slots), gpu.up(weights)
    dst, copy = gpu.out(m * n), gpu.out(m * n)
    gpu.call("ughip_add_rms_norm_rows", view(sx, 0, n), view(sy, 0, n), p(ss), p(swt), Z(top), Z(rows), p(sw), C.c_float(eps), View(None, 0, 0), view(dst, 0, n), p(sn) if second else None,
             p(copy), Z(m), Z(n))
    close(get(dst, (m, n)), want, 5e-6)
    close(get(copy, (m, n)), ph.rms(want, eps) * nxt if second else want, 8e-6)


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("t, want", [(40, [39]), (40, [7, 0, 39]), (3, [1, 1]), (2, [1, 0]), (130, list(range(129))), (1, [0])])
def test_llama_logits_of_some_positions(hip, bf16, t, want):
    """The head on the wanted rows alone gives what it gives among all of them, and the state behind the step is the same."""
    import ug_amd
    cfg = {"model_type": "llama", "hidden_size": 256, "intermediate_size": 512, "max_position_embeddings": 256, "num_attention_heads": 4, "num_key_value_heads": 2, "num_hidden_layers": 2,
           "rms_norm_eps": 1e-5, "vocab_size": 97}
    model = ug_amd.Decoder.random(hip, cfg, bf16=bf16, seed=3, std=0.1, norm_mean=1.0)
    tokens = np.random.default_rng(t).integers(0, 97, t)
    all_state, state = model.new_state(200), model.new_state(200)
    full, some = model.step(all_state, tokens, want=np.arange(t)), model.step(state, tokens, want=want)
    assert some.shape == (len(want), 97)
    np.testing.assert_allclose(some, full[want], rtol=0, atol=2e-5 * np.abs(full).max())   # the same f32 sums in another order
    np.testing.assert_array_equal(model.step(state, [5], want=[0]), model.step(all_state, [5], want=[0]))


# more chunks and heads than the chip has CUs, and half the heads of them at a time: two forms of the preparation, with 16-byte loads and without
@pytest.mark.parametrize("d, vd", [(64, 16), (100, 32), (99, 17), (128, 128)])
def test_delta_rows_of_many_heads_and_of_half_of_them(hip, d, vd):
    """The rows of a head are the same bits whichever form prepares its chunks (and those of a few heads are held to float64 elsewhere)."""
    from gpu_calls import Delta
    gpu, H, T, eps = Gpu(hip), 172, 100, 1e-5
    q, k, v, a, z = (rand(i, T, H, n) for i, n in enumerate((d, d, vd, d, vd)))
    b, a_log, dt_bias, norm = rand(6, T, H), rand(7, H), rand(8, H, d), rand(9, vd) + 1

    def rows(heads):
        n = heads.stop - heads.start
        s = {"qkv": np.concatenate([x[:, heads].reshape(T, -1) for x in (q, k, v)], 1), "b": b[:, heads], "a": a[:, heads], "z": z[:, heads], "a_log": a_log[heads], "dt": dt_bias[heads], "norm": norm}
        s = {name: gpu.up(np.ascontiguousarray(x)) for name, x in s.items()}
        S, dst = gpu.out(n * d * vd), gpu.out(T * n * vd)
        print("delta rows", n, d, vd, flush=True)
        gpu.call("ughip_delta_rows", C.byref(Delta(t=T, pos=0, heads=n, kv_heads=n, dim=d, vdim=vd, a_log=s["a_log"].raw(), dt_bias=s["dt"].raw(), norm=s["norm"].raw(), s=S.raw(), eps=eps,
                                                   qkv=view(s["qkv"], 0, n * (2 * d + vd)), b=view(s["b"], 0, n), a=view(s["a"], 0, n * d), z=view(s["z"], 0, n * vd), dst=view(dst, 0, n * vd))))
        return get(dst, (T, n, vd)), get(S, (n, d, vd))

    whole, state = rows(slice(0, H))
    assert np.all(np.isfinite(whole)) and np.all(np.isfinite(state))
    for heads in (slice(0, 86), slice(86, 172)):
        part, part_state = rows(heads)
        np.testing.assert_array_equal(whole[:, heads], part)
        np.testing.assert_array_equal(state[heads], part_state)
