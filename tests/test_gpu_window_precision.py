"""GPU test of the one-pass window forward's precision where any length is allowed: no further from float64 than weights rounded against a
running maximum over 64-key tiles (what the general kernel does)."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


def _bf16(x):
    return x.float().to(torch.bfloat16).double()


@pytest.mark.parametrize("s,w,docs", [(1001, 128, None), (777, 64, None), (555, 96, None), (501, 32, None), (999, 128, (300, 95, 404, 200))])
def test_no_further_from_float64_than_a_running_maximum(A, s, w, docs):
    print(f"case S={s} W={w} docs={docs}", flush=True)
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(9700 + s, 1, 16, 2, s, 64, torch.bfloat16))
    ds = torch.tensor([[sum(docs[:i]) for i, n in enumerate(docs) for _ in range(n)]], dtype=torch.int32, device=DEV) if docs else None
    o, _ = A.attention_forward(q, k, v, sinks, SCALE, w, 0, None, ds)
    i, j = torch.arange(s, device=DEV)[:, None], torch.arange(s, device=DEV)[None]
    seen = (j <= i) & (j > i - w)
    if docs:
        seen &= j >= ds[0, :, None]
    exact, running = (torch.empty(s, 16, 64, dtype=torch.float64, device=DEV) for _ in range(2))
    for h in range(16):
        keys, values = k[0, h // 8].double(), v[0, h // 8].double()
        logits = (q[0, h].double() @ keys.T * SCALE).masked_fill(~seen, -torch.inf)
        top = torch.maximum(logits.max(1).values, sinks[h].double())
        z = torch.exp(logits - top[:, None]).sum(1) + torch.exp(sinks[h].double() - top)
        exact[:, h] = torch.exp(logits - top[:, None]) @ values / z[:, None]
        m, acc = sinks[h].double().expand(s), torch.zeros(s, 64, dtype=torch.float64, device=DEV)
        for n in range(0, s, 64):
            m_new = torch.maximum(m, logits[:, n:n + 64].max(1).values)
            acc = acc * torch.exp(m - m_new)[:, None] + _bf16(torch.exp(logits[:, n:n + 64] - m_new[:, None])) @ values[n:n + 64]
            m = m_new
        running[:, h] = _bf16(acc / (z * torch.exp(top - m))[:, None])
    error, limit = (float((x - exact).norm() / exact.norm()) for x in (o[0].double(), running))
    assert error <= limit, (error, limit)
