"""Models whose decode steps make the output projection in attention's launch or in the one that merges its items: the plain model's logits, and
replayed steps with the bits of eager ones."""

import numpy as np
import pytest
import torch

import helpers
import plain_qwen2 as plain

pytestmark = pytest.mark.gpu

# the 0.5B shape's attention and width (14 heads on 2 of 64: steps of one to four requests take the joined launches), two small layers
NARROW = {
    "architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "hidden_size": 896, "num_hidden_layers": 2, "num_attention_heads": 14,
    "num_key_value_heads": 2, "head_dim": 64, "intermediate_size": 256, "vocab_size": 331, "rope_theta": 1000000.0, "rms_norm_eps": 1e-6,
    "tie_word_embeddings": True, "max_position_embeddings": 8192, "use_sliding_window": False,
}


@pytest.fixture(scope="module")
def folder(tmp_path_factory):
    return helpers.make_model_dir(tmp_path_factory.mktemp("narrow") / "m", NARROW, seed=91)


class Counted:
    """The calls of the joined launches, and of the merge by itself."""

    def __init__(self, monkeypatch):
        from from_scratch_inference_engine_amd import ops

        self.clear()
        qkv, merge_o, merge = ops.attention_mfma_qkv, ops.attention_merge_o, ops.attention_merge

        def run_qkv(*a, **k):
            self.whole += k.get("o_weight") is not None
            return qkv(*a, **k)

        def run_merge_o(*a, **k):
            self.merged += 1
            return merge_o(*a, **k)

        def run_merge(*a, **k):
            self.apart += 1
            return merge(*a, **k)

        monkeypatch.setattr(ops, "attention_mfma_qkv", run_qkv)
        monkeypatch.setattr(ops, "attention_merge_o", run_merge_o)
        monkeypatch.setattr(ops, "attention_merge", run_merge)

    def clear(self):
        self.whole = self.merged = self.apart = 0

    def only(self, way):
        mine = getattr(self, way)
        return 0 < mine == sum(vars(self).values())


def decode(runner, prompts, feed, steps):
    """The logits of ``steps`` tokens behind the prompts, one tensor a step."""
    from from_scratch_inference_engine_amd.engine.context import StepEntry

    caches = [runner.manager.open(i) for i in range(len(prompts))]
    runner.step([StepEntry(c, p, []) for c, p in zip(caches, prompts)])
    out = [runner.step([StepEntry(c, [f[t]], [0]) for c, f in zip(caches, feed)]).clone() for t in range(steps)]
    for c in caches:
        runner.manager.close(c)
    return out


@pytest.mark.parametrize("dtype, lengths, joined", [
    ("bfloat16", [40], "whole"), ("bfloat16", [60, 31], "whole"), ("bfloat16", [300], "merged"), ("bfloat16", [60, 400], "merged"),
    ("bfloat16", [600, 40], "merged"), ("bfloat16", [350, 20, 500], "merged"), ("bfloat16", [2000, 40, 40], "merged"),
    ("bfloat16", [40, 127, 214, 301], "merged"),
    ("float32", [300], "merged"), ("float32", [600, 40], "merged"), ("float32", [40, 127, 214, 301], "merged"),
])
def test_replays_have_the_bits_of_eager_steps(folder, dtype, lengths, joined, monkeypatch):
    """A shape runs eagerly the first times it comes and as a replayed graph from then on: whether the output projection is joined, and so the order of its
    sums, must not follow from that, also where some requests are whole and others cut (the graph merges every row, an eager step the cut ones)."""
    from from_scratch_inference_engine_amd import load_model
    from from_scratch_inference_engine_amd.engine.model import Runner

    model = load_model(folder, dtype=dtype)
    prompts = [helpers.token_ids(331, n, 60 + n) for n in lengths]
    feed = [helpers.token_ids(331, 4, 70 + n) for n in lengths]
    seen, calls = [], Counted(monkeypatch)
    for graphs in (False, True):
        runner = Runner(model, page_size=16, num_pages=sum(n // 16 + 2 for n in lengths) + 4, max_requests=4, use_graphs=graphs)
        calls.clear()
        seen.append(decode(runner, prompts, feed, 4))
        print(f"graphs {graphs}: {vars(calls)}")
        if graphs:
            assert runner.graphs.captures == 1 and runner.graphs.replays == 3
    for t, (a, b) in enumerate(zip(*seen)):
        assert torch.equal(a, b), f"step {t}"
    assert calls.only(joined)


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("dtype, lengths, way", [
    ("bfloat16", [29], "whole"), ("bfloat16", [29, 62], "whole"), ("bfloat16", [310], "merged"), ("bfloat16", [12, 420, 15], "merged"),
    ("float32", [140], "merged"), ("float32", [12, 420, 15], "merged"), ("float32", [2200], "apart"),  # (35 records)
])
def test_plain_logits_and_nan_in_the_pools(folder, dtype, lengths, way, graphs, monkeypatch):
    """Every page holds NaN, as an earlier request whose activations overflowed leaves it; decoding crosses the edges of pages, where many workgroups
    read the lines around a new key and value that one of them writes.  The logits are the plain model's."""
    from from_scratch_inference_engine_amd import load_model
    from from_scratch_inference_engine_amd.engine.model import Runner

    model, calls, steps = load_model(folder, dtype=dtype), Counted(monkeypatch), 6
    tokens = [helpers.token_ids(331, n + steps, 80 + n) for n in lengths]
    refs = [plain.forward_dir(folder, ids).numpy() for ids in tokens]
    runner = Runner(model, page_size=16, num_pages=sum(n // 16 + 2 for n in lengths), max_requests=4, use_graphs=graphs)
    k, v, _ = runner.storage.group_stores[0]
    k[:, 1:] = float("nan")
    v[:, 1:] = float("nan")
    out = decode(runner, [ids[:n] for ids, n in zip(tokens, lengths)], [ids[n:] for ids, n in zip(tokens, lengths)], steps)
    for i, n in enumerate(lengths):
        got = np.stack([o[i].float().cpu().numpy() for o in out])
        helpers.assert_close_to_plain(got, refs[i][n:n + steps], dtype, f"request {i} behind {n} tokens")
    assert calls.only(way), vars(calls)
    assert (k[:, 0] == 0).all() and (v[:, 0] == 0).all()
