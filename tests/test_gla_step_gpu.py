"""A step of one token a request of gated linear attention in one launch, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from from_scratch_inference_engine_amd import ops as module

    module.load(build_if_missing=False)
    return module


# every height and width of a head that the kernel takes; a bottleneck of one eight, of one round of the threads, of more than one
@pytest.mark.parametrize("heads, dim, vdim, rank", [(1, 16, 64, 8), (3, 32, 128, 24), (8, 128, 256, 64), (2, 256, 256, 136), (5, 64, 64, 72), (2, 128, 128, 128)])
def test_gla_step(ops, heads, dim, vdim, rank):
    assert ops.gla_step_takes(heads, dim, vdim, rank)
    gen = torch.Generator().manual_seed(heads * dim + rank)
    rnd = lambda *s: torch.randn(s, generator=gen)  # noqa: E731
    kw, vw, n_slots, tau, eps = heads * dim, heads * vdim, 7, 16.0, 1e-5
    # five requests: the third brings two tokens and the fourth has no slot, so both are left alone
    starts, slots = torch.tensor([0, 1, 2, 4, 5, 6], dtype=torch.int32), torch.tensor([4, 0, 2, -1, 6], dtype=torch.int32)
    g_off, a_off = 8 + 2 * kw + vw, 8 + 2 * kw + 2 * vw
    proj, a2, bias = rnd(6, a_off + rank).to(torch.bfloat16), (rnd(kw, rank) * rank ** -0.5).to(torch.bfloat16), 2.0 + 2.0 * rnd(kw)
    state, norm = rnd(n_slots, heads, dim, vdim), 1.0 + 0.3 * rnd(vdim)
    got_state = state.cuda()
    got = ops.gla_step(proj.cuda(), 8, 8 + kw, 8 + 2 * kw, g_off, a_off, a2.cuda(), bias.cuda(), got_state, starts.cuda(), slots.cuda(),
                       norm.cuda(), heads, dim, vdim, dim ** -0.5, 1.0 / tau, eps, "silu").cpu()
    p, want_state = proj.double(), state.double()
    for r, t in ((0, 0), (1, 1), (4, 5)):
        z = a2.double() @ p[t, a_off:] + bias.double()
        alpha = torch.sigmoid(z).pow(1.0 / tau).reshape(heads, dim)
        q, k = (p[t, at:at + kw].reshape(heads, dim) for at in (8, 8 + kw))
        v, g = (p[t, at:at + vw].reshape(heads, vdim) for at in (8 + 2 * kw, g_off))
        s = alpha.unsqueeze(-1) * want_state[slots[r]] + k.unsqueeze(-1) * v.unsqueeze(-2)
        want_state[slots[r]] = s
        o = (s * q.unsqueeze(-1)).sum(1) * dim ** -0.5
        y = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * norm.double() * g * torch.sigmoid(g)
        # one rounding to bfloat16 on float32 sums over the head's channels, which are of one size
        assert ((got[t].double().reshape(heads, vdim) - y).abs() <= 2.0 ** -8 * y.abs() + 1e-5 * y.abs().max()).all(), r
    assert ((got_state.cpu().double() - want_state).abs() <= 1e-5 * want_state.abs().max()).all()
    for slot in (1, 2, 3, 5):
        assert torch.equal(got_state[slot].cpu(), state[slot]), "a state that no request of one token owns"


def test_sizes_that_go_the_long_way(ops):
    for sizes in ((8, 48, 256, 64), (8, 128, 96, 64), (8, 128, 256, 12), (8, 128, 512, 64)):
        assert not ops.gla_step_takes(*sizes)


def test_one_projection_and_its_views(ops):
    """The weights become views of one matrix and the copy of the first a view of the whole's; a weight set anew undoes that."""
    from from_scratch_inference_engine_amd.parts.linear import Linear
    from from_scratch_inference_engine_amd.parts.linear_attention import GatedLinearAttention

    mixer = GatedLinearAttention(256, 2, 32, 64, 8, 16.0, 1e-5)
    gen = torch.Generator().manual_seed(1)
    w, a1 = (torch.randn(s, generator=gen).to(torch.bfloat16).cuda() for s in ((384, 256), (8, 256)))
    copies_from, Linear.streamed_copy_from = Linear.streamed_copy_from, 0
    try:
        mixer.qkvg_weight, mixer.a1_weight = w, a1
        mixer.o_weight = torch.zeros((256, 128), dtype=torch.bfloat16, device="cuda")
        mixer.prepare(torch.device("cuda"), torch.bfloat16)
    finally:
        Linear.streamed_copy_from = copies_from
    assert torch.equal(mixer.in_proj.weight, torch.cat([w, a1])) and torch.equal(mixer.qkvg_weight, w) and torch.equal(mixer.a1_weight, a1)
    assert mixer.a1_weight.data_ptr() == mixer.qkvg_weight.data_ptr() + w.numel() * 2
    assert torch.equal(mixer.qkvg.streamed.data, ops.fragment_order(w).data)
    assert mixer.release_optional_memory() == (392 + 8 + 256 * 128 // 256) * 256 * 2 and mixer.qkvg.streamed is None  # (392 rows: 400 in whole blocks)
    mixer.a1_weight = a1
    assert mixer.in_proj is None
