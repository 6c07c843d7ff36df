"""The prefill attention on the float32 matrix cores against the decode step:
a prompt prefilled in batches leaves the same logits, bit for bit, as one
decode step per token, at the edges of its tiles (16 rows of token x head, 64
positions, blocks of several tiles) and with positions of K or V that are not
finite."""
import os
import subprocess

import pytest
import torch

from tests.conftest import ROOT
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


@pytest.mark.parametrize("max_seq,n", [(4300, 4150), (262144, 800)])
def test_prefill_attention_three_passes(gpu, max_seq, n):
    """Passes that start past the prompt's first: 2048 + 2048 + 53 tokens, and four
    of at most 248, as many as 4096 splits' partials leave below 2 GB (which also
    takes the split combine that has no room for the weights of all splits)."""
    from spbitnet_amd.model import InferenceEngine, Model
    cfg = _small_config(max_position_embeddings=max_seq, num_key_value_heads=1)
    model = Model.random(cfg, seed=n)
    for lin in ("q_proj", "k_proj"):
        for l in model.layers:
            getattr(l, lin).gamma *= 0.05
    eng = InferenceEngine(model, max_seq=max_seq)
    out = []
    for batch in (1, 0):
        eng.set_prefill_batch(batch)
        eng.generate(_prompt(n, cfg.vocab_size, n), 1, stop_at_eos=False)
        out.append([_last_logits(eng)] + [c[:, :n].clone() for c in eng.kv_cache(1)])
        print(f"max_seq={max_seq} n={n} batch={batch}", flush=True)
    eng.close()
    assert torch.isfinite(out[1][0]).all()
    for got, want in zip(*out):
        assert torch.equal(got, want)


def test_mfma_is_a_chain_of_fused_multiply_adds(gpu):
    """What the kernel's equality rests on (tests/cpp/mfma_chain.hip, built by
    __graft_entry__.build())."""
    exe = os.path.join(ROOT, "tests", "cpp", "mfma_chain")
    assert os.path.exists(exe), "tests/cpp/mfma_chain is not built"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout, flush=True)
    assert r.returncode == 0, r.stdout + r.stderr


def _dense_row(lin, row):
    """Row `row` of a packed matrix as {-1, 0, 1} floats."""
    from spbitnet_amd import kernels as K
    dense = torch.empty((lin.rows, lin.cols), dtype=torch.int8, device="cuda")
    K.sparse_ternary_unpack_gpu(lin.meta, lin.values, dense, lin.rows, lin.cols, lin.meta_stride,
                                lin.values_stride)
    return dense[row].float()


@pytest.mark.parametrize("which", ["v", "k"])
@pytest.mark.parametrize("hd,nkv", [(64, 1), (128, 2)])
def test_prefill_attention_non_finite_positions(gpu, hd, nkv, which):
    """A position whose V (or K) is infinite leaves the tokens before it alone:
    it is not theirs to see, and a weight of 0 times infinity would be NaN.  The
    first layer's attention of those tokens shows in the second layer's K and V
    rows, which have to be finite and those of one decode step per token, bit for
    bit.  One token's embedding is a row of the projection, so that its product is
    some 20 times the others' spread and it alone passes the largest float."""
    from spbitnet_amd.model import InferenceEngine, Model
    cfg = _small_config(num_key_value_heads=nkv, head_dim=hd, hidden_size=8 * hd)
    model = Model.random(cfg, seed=hd + nkv)
    first, H = model.layers[0], cfg.hidden_size
    for lin in ("q_proj", "k_proj"):
        for l in model.layers:
            getattr(l, lin).gamma *= 0.05
    big = 7  # the token
    lin = first.v_proj if which == "v" else first.k_proj
    model.embed_tokens[big] = 0.02 * _dense_row(lin, 0).to(torch.bfloat16)
    first.input_layernorm.fill_(1.0)
    # the token's row is H / 2 values of sqrt(2), all quantised to 127: its product
    # is gamma * H / 2 * sqrt(2), 1.1 times the largest float
    lin.gamma = 1.1 * 3.4e38 / (H / 2 * 2 ** 0.5)
    if which == "v":
        first.o_proj.gamma *= 1e-37  # outputs of the usual size
    else:
        first.q_proj.gamma *= 1e-36  # scores of a few units
    eng = InferenceEngine(model, max_seq=256)
    # the only split of the prompt; its second split, of 36 positions; its third
    for at, n in ((21, 40), (70, 100), (150, 170)):
        prompt = [t if t != big else 8 for t in _prompt(n, cfg.vocab_size, n)]
        prompt[at] = big
        rows, logits = [], []
        for batch in (1, 0):
            eng.set_prefill_batch(batch)
            eng.generate(prompt, 1, stop_at_eos=False)
            logits.append(_last_logits(eng))
            k0, v0 = eng.kv_cache(0)
            assert not (v0 if which == "v" else k0)[:, at].isfinite().all()
            assert (v0 if which == "v" else k0)[:, :at].isfinite().all()
            rows.append(torch.cat([c[:, :at] for c in (k0, v0, *eng.kv_cache(1))]))
        assert rows[1].isfinite().all(), (at, n)
        assert torch.equal(rows[0].view(torch.int16), rows[1].view(torch.int16)), (at, n)
        same = logits[0].view(torch.int32) == logits[1].view(torch.int32)
        assert (same | (logits[0].isnan() & logits[1].isnan())).all()
    eng.close()


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
