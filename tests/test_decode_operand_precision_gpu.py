"""What the decode attention's matrix-pipe form makes of its fp32 operands: q rows of any finite size, and
softmax weights far below a row's largest, against float64 and against the shape-agnostic kernel, which
multiplies plain fp32 numbers."""
import numpy as np
import pytest

from paged_cases import DeviceCase, make_case

pytestmark = pytest.mark.gpu


def _exact(c):
    """softmax(q.K / sqrt(D)).V in float64, [batch, heads, D], from the values the call is given."""
    G, D = c.num_heads // c.kv_heads, c.head_dim
    pools = [p.view(np.float16).reshape(c.capacity_pages, c.page_size, c.kv_heads, D) for p in (c.k_pages, c.v_pages)]
    out = np.zeros((c.batch, c.num_heads, D))
    for r in range(c.batch):
        n = int(c.seq_lens[r])
        ids = c.page_tables_flat[c.page_table_offsets[r]:c.page_table_offsets[r + 1]]
        k, v = (p[ids].reshape(-1, c.kv_heads, D)[:n].astype(np.float64) for p in pools)
        for h in range(c.num_heads):
            s = k[:, h // G] @ c.q[r, h].astype(np.float64) / np.sqrt(D)
            w = np.exp(s - s.max())
            out[r, h] = (w / w.sum()) @ v[:, h // G]
    return out


def _run(exe, c, **options):
    dev = DeviceCase(exe, c)
    try:
        for name, value in options.items():
            assert exe.setOption(name, value)
        return dev.run().astype(np.float64), exe.lastDecodeKernel()
    finally:
        for name in options:
            exe.setOption(name, 0)
        dev.free()


def _errors(got, want):
    """2-norm and largest error of the whole output, both over its root mean square."""
    rms = np.sqrt(np.mean(want ** 2))
    return np.sqrt(np.mean((got - want) ** 2)) / rms, np.max(np.abs(got - want)) / rms


@pytest.mark.parametrize("D,P", [(64, 64), (64, 16), (128, 64), (128, 8)])
@pytest.mark.parametrize("ratio", [3, 4, 6, 8, 16])
def test_q_of_any_finite_size(exe, D, P, ratio):
    """Heads of 1e6 and of 1e-6 side by side over keys of 2e4, a head of zeros, one with an infinite element."""
    c = make_case(f"q_{ratio}_{D}_{P}", 3, 2 * ratio, 2, D, P, [40, 300, 777], seed=ratio + D + P)
    k = c.k_pages.view(np.float16)
    k *= np.float16(2e4 / 6)                    # (the largest of these normal values is below 6)
    c.q *= np.where(np.arange(2 * ratio) % 2, 1e-6, 1e6).astype(np.float32)[None, :, None]
    c.q[0, 1] = 0.0
    want = _exact(c)
    c.q[1, 0, 5] = np.inf
    got, kernel = _run(exe, c)
    assert "mfma" in kernel, kernel
    plain, _ = _run(exe, c, decode_force_generic=1)
    keep = np.ones(c.q.shape[:2], bool)
    keep[1, 0] = False                          # (what an infinite q gives is not defined; the others must not notice)
    assert np.isfinite(got[keep]).all()
    for big in (0, 1):                          # the two sizes apart: neither hides the other's error
        sel = keep & (np.arange(2 * ratio) % 2 == big)[None, :]
        e, p = _errors(got[sel], want[sel])[0], _errors(plain[sel], want[sel])[0]
        assert e <= p + 2.0 ** -22, (big, e, p)  # (a result is stored with an error of 2^-24 of itself)


@pytest.mark.parametrize("D,P", [(64, 64), (64, 16), (128, 64), (128, 16)])
@pytest.mark.parametrize("ratio", [3, 4, 6, 8, 16])
@pytest.mark.parametrize("outliers", [0.0, 0.01])
def test_error_is_no_larger_than_with_fp32_operands(exe, D, P, ratio, outliers):
    c = make_case(f"e_{ratio}_{D}_{P}", 4, 4 * ratio, 4, D, P, [100, 900, 2000, 3000], seed=ratio + D + P, scale_k_rows=outliers)
    want = _exact(c)
    got, kernel = _run(exe, c)
    assert "mfma-p32" in kernel, kernel
    plain, name = _run(exe, c, decode_force_generic=1)
    assert name == "generic"
    (e, e_max), (p, p_max) = _errors(got, want), _errors(plain, want)
    print(f"[error] ratio {ratio} D {D} P {P} outliers {outliers}: {e:.2e} (max {e_max:.1e}), fp32 operands {p:.2e} ({p_max:.1e})")
    # The single largest error: an element of q is off by at most 2^-23 of itself where fp32 arithmetic, which
    # rounds its product with the softmax scale, is off by at most 2^-24: at most twice as far.
    assert e <= p and e_max <= 2 * p_max


@pytest.mark.parametrize("D", [64, 128])
def test_small_weights_keep_their_bits(exe, D):
    """V is the unit matrix, so the output is the softmax weights: each to 2e-5 of itself down to 2^-12 of the
    row's largest, a few ulp of a score sum of 64 (64 * 2^-24 * ln 2 = 2.6e-6 each).  (A weight held as an fp16
    number and a remainder without a scale of its own is wrong by 2^-25 of the reference: 1e-4 of it there.)"""
    c = make_case(f"w_{D}", 24, 32, 4, D, 64, [D] * 24, seed=D, scale_k_rows=0.02, permute=False)
    c.v_pages.view(np.float16).reshape(24, D, 4, D)[...] = np.eye(D)[None, :, None, :]
    want = _exact(c)
    got, kernel = _run(exe, c)
    assert "mfma-p32" in kernel, kernel
    seen = want >= want.max(axis=2, keepdims=True) * 2.0 ** -12
    assert (want[seen] < 2.0 ** -10).sum() > 1000
    rel = np.abs(got[seen] / want[seen] - 1.0)
    assert rel.max() <= 2e-5, rel.max()
