"""The product of up to 16 rows whose K is under way at once: against float64, at the edges of its blocks, steps and slices."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from from_scratch_inference_engine_amd import ops as module

    module.load(build_if_missing=False)
    return module


def operands(m, n, k):
    gen = torch.Generator().manual_seed(1000 * m + n + k)
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16).cuda() for s in ((m, k), (n, k)))
    exact, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    return x, w, exact, k * 2.0 ** -24 * size  # a float32 rounding for each of K additions of each term


# one step of K; a step fewer and more than the waves hold evenly; the most a workgroup of 4, 8 and 16 waves holds; N that ends inside
# a block of 16 rows and inside a pair of blocks
@pytest.mark.parametrize("m, n, k", [(1, 4, 32), (16, 36, 96), (3, 52, 1024), (7, 1168, 1056), (16, 80, 2048), (2, 20, 2080), (9, 100, 4064), (16, 48, 4096)])
@pytest.mark.parametrize("frags", [True, False])
def test_whole_products(ops, m, n, k, frags):
    x, w, exact, bound = operands(m, n, k)
    weight, bias = ops.fragment_order(w) if frags else w, torch.randn(n, generator=torch.Generator().manual_seed(n)).cuda()
    steps = k // 32
    for waves in (4, 8, 16):
        for blocks in (1, 2):
            if -(-steps // waves) > 8 or (waves == 4 and blocks == 2):
                continue
            got = ops.gemm_mfma_stream(x, weight, ops.GEMM_STREAM_POINT, waves + 256 * blocks + 65536, bias).double()
            want = exact + bias.double()
            assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2 * bound).all(), (waves, blocks)  # one rounding to bfloat16
            if frags:
                got = ops.gemm_mfma_stream(x, weight, ops.GEMM_STREAM_GATED, waves + 256 * blocks + 65536, act="relu").double()
                gate, up = exact[:, 0::2], exact[:, 1::2]
                want, off = gate.clamp(min=0) * up, bound[:, 0::2] * up.abs() + bound[:, 1::2] * gate.abs()
                assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2 * off).all(), (waves, blocks)


@pytest.mark.parametrize("m, n, k, splits", [(1, 17, 1024, 1), (16, 33, 2048, 2), (5, 896, 4864, 4), (8, 31, 4864, 3), (16, 1536, 8960, 5), (2, 100, 1056, 2)])
def test_partial_sums(ops, m, n, k, splits):
    x, w, exact, bound = operands(m, n, k)
    f = ops.fragment_order(w)
    for blocks in (1, 2):
        got = ops.gemm_mfma_stream(x, f, ops.GEMM_STREAM_SUMS, 8 + 256 * blocks + 65536 * splits)
        assert got.shape == (splits, m, n) and got.dtype == torch.float32
        assert ((got.double().sum(0) - exact).abs() <= bound).all(), blocks
    k_slice = -(-(k // 32) // splits) * 32  # a slice holds its own part of K only
    first = x[:, :k_slice].double() @ w[:, :k_slice].double().t()
    assert ((got[0].double() - first).abs() <= bound).all()


def test_what_the_plan_takes(ops):
    """A plan is one the kernel takes; where it stops: rows, K, steps of K, and for one or two rows the widest gate and up matrices."""
    if ops.compute_units() != 256:
        pytest.skip("the figures are those of 256 units")
    plan = ops.gemm_stream_plan
    assert plan(8, 896, 4864, ops.GEMM_STREAM_SUMS, True) == 8 + 256 + 4 * 65536
    assert plan(8, 2048, 8192, ops.GEMM_STREAM_SUMS, True) == 8 + 512 + 4 * 65536
    assert plan(8, 3584, 3584, ops.GEMM_STREAM_SUMS, True) == 8 + 512 + 2 * 65536
    for n, k, frags in ((3584, 18944, True), (4608, 3584, True), (896, 896, True), (896, 4864, False)):
        assert plan(8, n, k, ops.GEMM_STREAM_SUMS, frags) is None
    assert plan(8, 9728, 896, ops.GEMM_STREAM_GATED, True) == 4 + 256 + 65536 and plan(9, 9728, 896, ops.GEMM_STREAM_GATED, True) is None
    assert plan(16, 8192, 1024, ops.GEMM_STREAM_GATED, True) and plan(2, 22016, 2048, ops.GEMM_STREAM_GATED, True) is None
    assert plan(4, 14336, 4096, ops.GEMM_STREAM_PLAN_ACT, True) and plan(5, 14336, 4096, ops.GEMM_STREAM_PLAN_ACT, True) is None
    assert plan(5, 14336, 4096, ops.GEMM_STREAM_POINT, True) and plan(5, 4112, 896, ops.GEMM_STREAM_POINT, False) is None
    assert plan(2, 16384, 2048, ops.GEMM_STREAM_GATED, True) and plan(3, 16384, 2048, ops.GEMM_STREAM_GATED, True) is None
    assert plan(17, 896, 896, ops.GEMM_STREAM_POINT, True) is None and plan(0, 896, 896, ops.GEMM_STREAM_POINT, True) is None
    assert plan(8, 896, 4128, ops.GEMM_STREAM_POINT, True) is None and plan(8, 898, 896, ops.GEMM_STREAM_POINT, True) is None
    x = torch.zeros((4, 100), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ops.KernelError, match="bad sizes"):
        ops.gemm_mfma_stream(x, torch.zeros((8, 100), dtype=torch.bfloat16, device="cuda"), ops.GEMM_STREAM_POINT, 4 + 256 + 65536)


def test_the_largest_weights_in_rows_take_up_to_eight_rows(ops):
    if ops.compute_units() != 256:
        pytest.skip("the figures are those of 256 units")
    plan = ops.gemm_stream_plan
    for result in (ops.GEMM_STREAM_POINT, ops.GEMM_STREAM_PLAN_ACT):
        assert plan(8, 4096, 4096, result, False) and plan(9, 4096, 4096, result, False) is None
        assert plan(16, 3584, 3584, result, False) and plan(16, 4096, 4096, result, True)


def test_every_plan_is_one_that_the_kernel_takes(ops):
    """Over sizes of all kinds, K beyond what sixteen slices hold among them: the checks of the launch itself, and the residual
    projections of such sizes."""
    from from_scratch_inference_engine_amd.parts.linear import Linear

    taken = {r: 0 for r in range(4)}
    for k in [32 * s for s in (1, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 152, 511, 512, 513, 592, 1023, 1024, 1025, 1152, 1280, 2048)]:
        for n in (4, 16, 20, 36, 64, 100, 256, 272, 896, 1536, 2048, 3584, 4096, 4112, 8192, 11264, 19456, 37888):
            for result in taken:
                for m in (1, 2, 3, 8, 9, 16):
                    for frags in (True, False):
                        plan = ops.gemm_stream_plan(m, n, k, result, frags)
                        if plan is None:
                            continue
                        taken[result] += 1
                        waves, blocks, splits = plan & 255, plan >> 8 & 255, plan >> 16
                        slice_steps = -(-(k // 32) // splits)
                        assert 1 <= splits <= (16 if result == ops.GEMM_STREAM_SUMS else 1) and slice_steps * (splits - 1) < k // 32, (m, n, k, result)
                        assert waves in (4, 8, 16) and blocks in (1, 2) and -(-slice_steps // waves) <= 8, (m, n, k, result)
                        assert frags or result in (ops.GEMM_STREAM_POINT, ops.GEMM_STREAM_PLAN_ACT)
                        # (one of the kernels that are compiled as it is, none rounded up)
                        assert -(-slice_steps // waves) >= {4: 1, 8: 4 if result == ops.GEMM_STREAM_SUMS else 5, 16: 5}[waves], (m, n, k, result)
                        assert blocks == 1 or (waves == 8 and frags), (m, n, k, result)
    assert min(taken.values()) > 100
    for n, k in ((256, 36864), (64, 40960)):
        x, w, exact, bound = operands(8, n, k)
        linear = Linear(k, n)
        linear.weight = w
        linear.streamed = ops.fragment_order(w)
        sums = linear.for_residual(x, type("Step", (), {"partial_sums_ok": True}))
        got = (sums.double().sum(0) if sums.dim() == 3 else sums.double())
        assert ((got - exact).abs() <= bound + (0 if sums.dim() == 3 else 2.0 ** -8 * exact.abs())).all(), (n, k)


# a step of K in each half, as many as four and eight waves hold in 7, 8, 6 and 8 steps each and one fewer; N that ends inside a block of 16 rows;
# no, one, some and all partial sums that are asked for together
@pytest.mark.parametrize("m, n, k, parts", [(1, 4, 64, 0), (2, 36, 896, 1), (1, 1152, 896, 4), (2, 52, 864, 3), (1, 20, 1024, 8), (2, 100, 1536, 5), (1, 68, 2048, 7), (2, 48, 2016, 2)])
@pytest.mark.parametrize("frags", [True, False])
def test_a_norm_in_the_product_behind_it(ops, m, n, k, parts, frags):
    gen = torch.Generator().manual_seed(n + k + parts)
    rand = lambda *s: torch.randn(s, generator=gen).cuda()
    res, sums, nw, w = rand(m, k), rand(parts, m, k) if parts else None, 1 + 0.1 * rand(k), rand(n, k).to(torch.bfloat16)
    want_stream, old = res.clone(), res.clone()
    x = ops.rmsnorm(want_stream, nw, 1e-6, torch.bfloat16, delta=sums, write_back=parts > 0)
    exact, bound = x.double() @ w.double().t(), k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    weight = ops.fragment_order(w) if frags else w
    new = torch.full_like(res, float("nan"))
    for splits in (1, 2):
        got = ops.gemm_mfma_normed(res, sums, nw, 1e-6, new, weight, ops.GEMM_STREAM_SUMS, splits=splits)
        assert got.shape == (splits, m, n) and torch.equal(res, old)
        assert ((got.double().sum(0) - exact).abs() <= bound).all(), splits  # (the normed row is the norm kernel's, bit for bit)
    assert torch.equal(new, want_stream) if parts else new.isnan().all()
    gate, up = exact[:, 0::2], exact[:, 1::2]
    got = ops.gemm_mfma_normed(res, sums, nw, 1e-6, new, weight, ops.GEMM_STREAM_GATED, act="relu").double()
    want, off = gate.clamp(min=0) * up, bound[:, 0::2] * up.abs() + bound[:, 1::2] * gate.abs()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2 * off).all()


@pytest.mark.parametrize("heads, kv", [(4, 2), (8, 2)])
def test_steps_of_one_and_two_requests_leave_their_norms_to_the_products(heads, kv, monkeypatch):
    """Whole steps with and without, eager and replayed: the normed rows are the same bit for bit and the products' float32 sums
    are made in other slices, which may round to neighbouring bfloat16 values (2^-8 of a value) in each of the layers."""
    from from_scratch_inference_engine_amd import LLM
    from from_scratch_inference_engine_amd.engine.context import StepEntry
    from from_scratch_inference_engine_amd.ops import functions
    from from_scratch_inference_engine_amd.parts.block import PreNormBlock
    from from_scratch_inference_engine_amd.parts.linear import Linear

    monkeypatch.setattr(Linear, "streamed_copy_from", 1 << 19)
    raw = {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "hidden_size": 64 * heads * 2, "num_hidden_layers": 3,
           "num_attention_heads": heads, "num_key_value_heads": kv, "head_dim": 128, "intermediate_size": 1024, "vocab_size": 500,
           "rope_theta": 10000.0, "rms_norm_eps": 1e-6, "tie_word_embeddings": True, "max_position_embeddings": 512}
    seen, product = [], functions.gemm_mfma_normed
    counted = lambda *a, **k: (seen.append(a[0].shape[0]), product(*a, **k))[1]
    for module in ("ops", "ops.functions"):  # (q/k/v asks for it, gate and up come by their own name)
        monkeypatch.setattr(f"from_scratch_inference_engine_amd.{module}.gemm_mfma_normed", counted)
    out = {}
    for rows in (0, 2):
        monkeypatch.setattr(PreNormBlock, "few_rows", rows)
        llm = LLM.from_config(raw, weight_seed=3, block_size=16, num_blocks=64, max_batch=4, dtype="bfloat16")
        runner, steps = llm.engine.runner, []
        for n in (1, 2, 3):
            caches = [runner.manager.open((n, r)) for r in range(n)]
            runner.step([StepEntry(c, list(range(5 + r, 40 + 3 * r)), []) for r, c in enumerate(caches)])
            for t in range(7):  # (the third of a shape is captured, the others behind it replayed)
                steps.append(runner.step([StepEntry(c, [7 * t + r], [0]) for r, c in enumerate(caches)]))
            for c in caches:
                runner.manager.close(c)
        out[rows] = torch.cat(steps)
        assert (len(seen) == 0) if rows == 0 else (set(seen) == {1, 2} and len(seen) % 6 == 0)
    a, b = out[0].double(), out[2].double()
    assert ((a - b).norm(dim=1) <= 3 * 2 * 2.0 ** -8 * a.norm(dim=1)).all()
