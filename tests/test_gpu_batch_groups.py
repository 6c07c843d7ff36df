"""A batch whose positions pass from the step graphs with one sequence group to
those with two (768 positions) during a generation: every sequence's tokens
equal those of the single-sequence engine."""
import pytest

from tests.test_gpu_engine import _prompt, _small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [24, 32])
def test_batch_crosses_into_two_groups(gpu, batch):
    from spbitnet_amd.model import BatchInferenceEngine, InferenceEngine, Model
    cfg = _small_config(num_key_value_heads=2, max_position_embeddings=2048)
    model = Model.random(cfg, seed=batch)
    lens = [760 if i == batch - 1 else 5 + 23 * i for i in range(batch)]
    prompts = [_prompt(n, cfg.vocab_size, i) for i, n in enumerate(lens)]
    eng = BatchInferenceEngine(model, max_seq=1100, batch=batch)
    got = eng.generate(prompts, 20, stop_at_eos=False)
    eng.close()
    one = InferenceEngine(model, max_seq=1100)
    for i, p in enumerate(prompts):
        assert got[i] == one.generate(p, 20, stop_at_eos=False), i
    one.close()
