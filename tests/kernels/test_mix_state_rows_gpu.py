"""Recurrences of decode rows (csrc/kernels/mix_state_rows.hip) against the token-by-token reference: head sizes around
the eight lanes of a key group and the 32 value channels of a wave, states that begin and go on, lists of runs with
padding whose other entries hold longer runs, and operands that the kernel leaves to the general one."""
import pytest
import torch

from replisense_rfq_amd import ops
from replisense_rfq_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(lens, entries):
    rs, rb, rf, pos, runs = [], [], [], [], []
    for i, n in enumerate(lens):
        runs.append(len(rs))
        rs += [-1 if i == 3 else 2 * i + i % 2] * n
        rb += range(n)
        rf += range(n - 1, -1, -1)
        pos += range(17 * (i % 2), 17 * (i % 2) + n)
    runs = [-1] * (entries - len(runs)) + runs
    return [torch.tensor(x, dtype=torch.int32) for x in (rs, rb, rf, pos)], torch.tensor(runs, dtype=torch.int32)


def _near(got, want, tol, worst=8):
    got, want = got.double().cpu(), want.double()
    assert float((got - want).square().mean().sqrt()) <= tol * float(want.square().mean().sqrt())
    assert float((got - want).abs().max()) <= worst * tol * max(1.0, float(want.square().mean().sqrt()))


# a state's entry is a decay's product and one sum more a row, a read-out 128 products: a few units of 2^-24 each, the
# norm's division the same; bf16 read-outs are one rounding (2^-9) of that
# The worst entry of a read-out: a head's 64 terms may cancel, of the few dozen heads here to about a 64th of their sizes
# (in the kernel for 32 channels, 2.7e-5 for one head of wkv), and the norm divides by what is left.
WORST = 64
TOL = {torch.float32: 2e-6, torch.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("dtype,lens", [(torch.float32, [1] * 7), (torch.bfloat16, [1] * 7), (torch.float32, [1]),
                                        (torch.float32, [2, 1, 5, 1])])
@pytest.mark.parametrize("H,Hq,dim,vdim,pad", [(2, 2, 64, 128, 4), (4, 2, 32, 4, 0), (3, 3, 128, 36, 4), (1, 1, 64, 256, 0),
                                               (4, 1, 128, 64, 8), (2, 2, 64, 60, 4), (2, 2, 64, 32, 1), (2, 1, 48, 20, 0)])
@pytest.mark.parametrize("delta", [False, True])
def test_gated_rows(delta, H, Hq, dim, vdim, pad, dtype, lens):
    g = torch.Generator().manual_seed(dim + vdim)
    T = sum(lens)
    wide = torch.randn(T, 2 * Hq * dim + H * vdim + pad, generator=g)
    qk = wide[:, :2 * Hq * dim].unflatten(1, (2 * Hq, dim))
    qk /= qk.square().sum(-1, keepdim=True).sqrt()
    wide = wide.to(dtype)
    z, zb, rate = torch.randn(T, H * dim, generator=g), torch.randn(H * dim, generator=g), torch.rand(H, generator=g) + 0.1
    beta = torch.randn(T, H, generator=g).to(dtype) if delta else None
    gate, nw = torch.randn(T, H * vdim + pad, generator=g).to(dtype), torch.randn(vdim, generator=g)
    st = torch.randn(2 * len(lens), H, dim, vdim, generator=g) * 0.3
    rows, runs = _rows(lens, T)

    def call(dev, f, **more):
        m = lambda x: None if x is None else x.to(dev)  # noqa: E731
        w, s, out = m(wide), m(st).clone(), torch.zeros(T, H * vdim, dtype=dtype, device=dev)
        q, k = (w[:, i * Hq * dim:(i + 1) * Hq * dim].unflatten(1, (Hq, dim)) for i in (0, 1))
        v = w[:, 2 * Hq * dim:2 * Hq * dim + H * vdim].unflatten(1, (H, vdim))
        f(q, k, v, m(z), m(rate), m(zb), 1.0, m(beta), m(gate)[:, :H * vdim], delta, m(nw), 1e-5, dim ** -0.5, s,
          *(m(r) for r in rows), out, **more)
        return out, s

    (out, s), (out_w, s_w) = call(DEV, ops.gated_linear_recurrence, run_rows=runs.to(DEV)), call("cpu", ref.gated_linear_recurrence)
    _near(out, out_w, TOL[dtype], WORST)
    _near(s, s_w, TOL[torch.float32])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N", [64, 32])
@pytest.mark.parametrize("lens", [[1] * 7, [1], [2, 1, 5, 1]])
def test_wkv_rows(lens, N, dtype):
    H, T = 3, sum(lens)
    g = torch.Generator().manual_seed(N + T)
    r, k, v, zw, gate = (torch.randn(T, H * N, generator=g).to(dtype) for _ in range(5))
    w0, u, nw = torch.randn(H * N, generator=g) - 2, torch.randn(H, N, generator=g), torch.randn(H * N, generator=g)
    st = torch.randn(2 * len(lens), H, N, N, generator=g) * 0.3
    rows, runs = _rows(lens, T)

    def call(dev, f, **more):
        out, s = torch.zeros(T, H * N, dtype=dtype, device=dev), st.to(dev).clone()
        f(*(x.to(dev) for x in (r, k, v, zw, w0, u, gate, nw)), 1e-5, s, *(x.to(dev) for x in rows), out, **more)
        return out, s

    (out, s), (out_w, s_w) = call(DEV, ops.wkv_recurrence, run_rows=runs.to(DEV)), call("cpu", ref.wkv_recurrence)
    _near(out, out_w, TOL[dtype], WORST)
    _near(s, s_w, TOL[torch.float32])
