"""GPU: a FastDecoder reads the model's settings (the discretization, the final norm's eps) at each step;
refresh() is for weights only."""

import pytest
import torch

from ssm_scan.block import MambaLM
from ssm_scan.decode import FastDecoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["stack", "block"])
def test_settings_changed_after_the_decoder_was_built(dev, path):
    torch.manual_seed(1)
    model = MambaLM(n_layers=2).to(dev).eval()
    fast = FastDecoder(model, path=path)
    tok = torch.arange(4, device=dev)

    def step(decoder):
        states = model.init_state(4, 1, dev)
        for s in states:
            s.ssm.fill_(0.5)
            s.conv.fill_(0.25)
        return decoder.step(tok, states)

    first = step(fast)
    for blk in model.blocks:
        blk.mixer.discretization = "euler"
    model.norm_f.eps = 0.5
    got = step(fast)
    assert torch.equal(got, step(FastDecoder(model, path=path)))
    assert not torch.allclose(got, first, rtol=1e-3)
