"""GPU: KernelTimer's events enclose the launches alone -- nothing is allocated or cast between them --
one pair for every launch."""

import pytest
import torch

import ssm_scan
from ssm_scan import scan as S

pytestmark = pytest.mark.gpu


class _End:
    def __init__(self, event, done):
        self.event, self.done = event, done

    def record(self):
        self.event.record()
        self.done()


class _Counting(ssm_scan.KernelTimer):
    """Notes the caching allocator's count of allocations at both events of every launch."""

    def __init__(self):
        super().__init__()
        self.allocated = []

    def begin(self, name):
        count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
        end, at = super().begin(name), count()
        return _End(end, lambda: self.allocated.append((name, at, count())))


def test_events_enclose_the_launch(dev):
    g = torch.Generator(device=dev).manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, delta, A, Bm, Cm = r(2, 70, 64).bfloat16(), r(2, 70, 64).abs() * 0.1, -r(64, 16).abs(), r(2, 70, 16), r(2, 70, 16)
    a, b = r(1, 33, 70).sigmoid(), r(1, 33, 70)
    with _Counting() as t:
        leaves = [v.requires_grad_() for v in (x, delta, A, Bm, Cm)]
        y, last = ssm_scan.selective_scan_fn(*leaves, return_last_state=True)   # x is cast
        torch.autograd.grad(last.sum(), leaves)                               # dout is filled
        for scan in ("chunked", "sequential"):
            y, last = S.selective_scan(*leaves, scan=scan, d_block=40)          # two launches backward
            torch.autograd.grad(y.sum(), leaves)
        h = S.scan_chunked(a.requires_grad_(), b.requires_grad_())
        torch.autograd.grad(h, (a, b), r(1, 70, 33).transpose(1, 2))
        u, v = S.discretize(*(q.requires_grad_() for q in (delta, A, Bm, x)))
        torch.autograd.grad(u, (delta, A), torch.ones_like(u))
    names = ["ssm_fwd", "ssm_bwd"] + 2 * ["ssm_cscan_fwd", "ssm_cscan_bwd", "ssm_cscan_bwd"] + [
        "ssm_lscan", "ssm_lscan_bwd", "ssm_disc_fwd", "ssm_disc_bwd"]
    assert [n for n, _, _ in t.allocated] == names
    assert all(before == after for _, before, after in t.allocated), t.allocated
    times = t.times_ms()
    assert sorted(times) == sorted(set(names)) and sum(len(v) for v in times.values()) == len(names)
    assert all(ms > 0 for v in times.values() for ms in v)
