"""The prefill attention on the float32 matrix cores against the decode step:
a prompt prefilled in batches leaves the same logits, bit for bit, as one
decode step per token, at the edges of its tiles (16 rows of token x head, 64
positions, blocks of several tiles) and with values of V that are not finite."""
import pytest
import torch

from tests.test_gpu_engine import _last_logits, _prompt, _small_config

pytestmark = pytest.mark.gpu


def _both(model, max_seq, prompt):
    """The next token's logits after the batched and the stepwise prefill."""
    from spbitnet_amd.model import InferenceEngine
    eng = InferenceEngine(model, max_seq=max_seq)
    out = []
    for batch in (1, 0):
        eng.set_prefill_batch(batch)
        eng.generate(prompt, 1, stop_at_eos=False)
        out.append(_last_logits(eng))
    eng.close()
    return out


# (head_dim, kv heads of 8): GQA groups 1, 2, 4 and 8
@pytest.mark.parametrize("hd,nkv", [(64, 8), (64, 4), (64, 2), (64, 1),
                                    (128, 8), (128, 4), (128, 2), (128, 1)])
def test_prefill_attention_tile_edges(gpu, hd, nkv):
    from spbitnet_amd.model import Model
    cfg = _small_config(num_key_value_heads=nkv, head_dim=hd, hidden_size=8 * hd)
    model = Model.random(cfg, seed=hd + nkv)
    for lin in ("q_proj", "k_proj"):  # scores of a few units: every position weighs in
        for l in model.layers:
            getattr(l, lin).gamma *= 0.05
    # n - 1 tokens prefill: one token, one row tile, a split and a token more,
    # a block of several tiles, five splits with a partial last one
    for n in (2, 5, 18, 65, 66, 131, 322, 700):
        print(f"hd={hd} nkv={nkv} prompt={n}", flush=True)
        batched, stepwise = _both(model, 768, _prompt(n, cfg.vocab_size, n))
        assert torch.isfinite(stepwise).all()
        assert torch.equal(batched.view(torch.int32), stepwise.view(torch.int32)), n


@pytest.mark.parametrize("hd,nkv", [(64, 1), (128, 2)])
def test_prefill_attention_non_finite_values(gpu, hd, nkv):
    """An infinite V at a later position leaves earlier tokens alone (its
    weight is not 0 times infinity: the position is not theirs to see)."""
    from spbitnet_amd.model import Model
    cfg = _small_config(num_key_value_heads=nkv, head_dim=hd, hidden_size=8 * hd)
    model = Model.random(cfg, seed=hd + nkv)
    for lin in ("q_proj", "k_proj"):
        for l in model.layers:
            getattr(l, lin).gamma *= 0.05
    # products reach about 3000 (4 sigma over 512 or 1024 columns): the largest overflow
    model.layers[0].v_proj.gamma = 3e38 / 2000 * 127 / 4
    for n in (40, 100):
        batched, stepwise = _both(model, 256, _prompt(n, cfg.vocab_size, n))
        same = batched.view(torch.int32) == stepwise.view(torch.int32)
        assert (same | (batched.isnan() & stepwise.isnan())).all()


@pytest.mark.parametrize("hd,nkv", [(64, 4), (128, 1)])
def test_packed_prompts_match_single_sequences(gpu, hd, nkv):
    """Prompts of several sequences share prefill passes: tokens equal those of
    each sequence alone, with prompts of one token, of one tile and ones that a
    pass of 2048 tokens cuts in two."""
    from spbitnet_amd.model import BatchInferenceEngine, InferenceEngine, Model
    cfg = _small_config(num_key_value_heads=nkv, head_dim=hd, hidden_size=8 * hd,
                        max_position_embeddings=2048)
    model = Model.random(cfg, seed=hd + nkv)
    for lin in ("q_proj", "k_proj"):
        for l in model.layers:
            getattr(l, lin).gamma *= 0.05
    lens = [1, 2, 17, 66, 700, 5, 1, 1500, 130, 900]
    prompts = [_prompt(n, cfg.vocab_size, i) for i, n in enumerate(lens)]
    eng = BatchInferenceEngine(model, max_seq=1600, batch=12)
    got = eng.generate(prompts, 8, stop_at_eos=False)
    eng.close()
    one = InferenceEngine(model, max_seq=1600)
    one.set_prefill_batch(0)
    for i, p in enumerate(prompts):
        assert got[i] == one.generate(p, 8, stop_at_eos=False), lens[i]
    one.close()
