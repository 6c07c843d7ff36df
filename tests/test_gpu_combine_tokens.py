"""The split combine of a prefill pass of many tokens: the logits after a
prompt prefilled in batches equal, bit for bit, those of one decode step per
token, where heads do not fill a wave (256 / head_dim heads) and at the edges
of its batches of eight splits."""
import pytest
import torch

from tests.test_gpu_engine import _prompt, _small_config
from tests.test_gpu_prefill_attention import _both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,nh,nkv", [(64, 6, 3), (64, 8, 2), (128, 3, 3), (128, 4, 1)])
def test_combine_tokens(gpu, hd, nh, nkv):
    from spbitnet_amd.model import Model
    cfg = _small_config(num_attention_heads=nh, num_key_value_heads=nkv, head_dim=hd,
                        hidden_size=nh * hd, max_position_embeddings=2304)
    model = Model.random(cfg, seed=hd + nh)
    for lin in ("q_proj", "k_proj"):  # scores of a few units: every position weighs in
        for l in model.layers:
            getattr(l, lin).gamma *= 0.05
    # 9 splits (the first past the fold in the producer), 16 full ones, 17, and
    # 33 (more than a head has lanes)
    for n in (514, 1025, 1030, 2115):
        print(f"hd={hd} nh={nh} prompt={n}", flush=True)
        batched, stepwise = _both(model, 2304, _prompt(n, cfg.vocab_size, n))
        assert torch.isfinite(stepwise).all()
        assert torch.equal(batched.view(torch.int32), stepwise.view(torch.int32)), n
