"""K5 tree attention and the verify-subtree forward on the device.

K5 is a floating-point kernel: it is compared with a torch fp32 reference of
the same masked grouped-query attention (the math of transformers'
sdpa_attention_forward, which the reference's target uses).  The model-level
tests restate tests/gpu/test_eagle3_tree.py:1435-1530 (each tree node's
logits equal an independent causal decode of its path) on a bf16 offloaded
model, so the tolerance is bf16's rather than fp32's.
"""
import math

import pytest
import torch

from specfit_amd import ops
from specfit_amd.runtime import (TREE_ATTENTION, Eagle3DraftTree, build_offloaded_qwen3,
                                 register_tree_attention, synthetic_tree, verify_draft_tree)

pytestmark = pytest.mark.gpu


def _reference(q, k, v, mask, scale):
    """fp32 masked GQA attention: q [B,Hq,Q,D], k/v [B,Hkv,S,D], mask
    [B,1,Q,S] bool or None (causal aligned to the end)."""
    B, Hq, Q, D = q.shape
    Hkv, S = k.shape[1], k.shape[2]
    G = Hq // Hkv
    kf = k.float().repeat_interleave(G, dim=1)
    vf = v.float().repeat_interleave(G, dim=1)
    s = torch.matmul(q.float(), kf.transpose(-1, -2).contiguous()) * scale
    if mask is None:
        qi = torch.arange(Q, device=q.device)[:, None]
        si = torch.arange(S, device=q.device)[None, :]
        mask = (si <= S - Q + qi).view(1, 1, Q, S)
    s = s.masked_fill(~mask, float("-inf"))
    p = torch.softmax(s, dim=-1)
    p = torch.nan_to_num(p, nan=0.0)
    return torch.matmul(p, vf).transpose(1, 2)  # [B, Q, Hq, D]


def _check(out, ref):
    assert out.shape == ref.shape and out.dtype == torch.bfloat16
    err = (out.float() - ref).abs()
    scale = ref.abs().max().clamp_min(1e-6)
    assert (err.max() / scale).item() <= 1e-2, (err.max() / scale).item()
    assert torch.all(err <= 8e-3 * ref.abs() + 2e-3 * scale)


def _rand(shape, device, g, std=1.0):
    return (torch.randn(shape, generator=g) * std).to(torch.bfloat16).to(device)


def test_verification_shape_with_tree_mask(device):
    g = torch.Generator().manual_seed(11)
    tree = synthetic_tree(60, 6, seed=5, vocab=151936)
    base, Q, Hq, Hkv, D = 1024, 61, 32, 4, 128
    S = base + Q
    q = _rand((1, Q, Hq, D), device, g).transpose(1, 2)  # HF layout: a transposed view
    k = _rand((1, Hkv, S, D), device, g)
    v = _rand((1, Hkv, S, D), device, g)
    mask = tree.verification_attention_mask(base_kv_length=base, device=device)
    scale = D ** -0.5
    out = ops.tree_attention(q, k, v, mask, scale)
    _check(out, _reference(q, k, v, mask, scale))
    again = ops.tree_attention(q, k, v, mask, scale)
    assert torch.equal(out, again)  # run-to-run identical


@pytest.mark.parametrize("Hq,Hkv,D", [(4, 4, 8), (4, 2, 8), (8, 2, 64), (16, 4, 128),
                                      (16, 1, 128), (32, 4, 96), (8, 2, 256),
                                      (32, 4, 128), (8, 4, 64), (8, 4, 128), (32, 2, 64),
                                      (64, 4, 128)])  # the last: Qwen3-235B-A22B attention
@pytest.mark.parametrize("Q,S", [(1, 1), (1, 300), (7, 7), (61, 1085), (130, 130)])
def test_shapes_causal_and_masked(device, Hq, Hkv, D, Q, S):
    if D == 256 and Hq // Hkv > 4:
        pytest.skip("exceeds the kernel's LDS budget")
    g = torch.Generator().manual_seed(Hq * 1000 + D + Q + S)
    q = _rand((1, Hq, Q, D), device, g)
    k = _rand((1, Hkv, S, D), device, g)
    v = _rand((1, Hkv, S, D), device, g)
    scale = 1.0 / math.sqrt(D)
    _check(ops.tree_attention(q, k, v, None, scale), _reference(q, k, v, None, scale))
    gm = torch.Generator().manual_seed(S)
    mask = (torch.rand((1, 1, Q, S), generator=gm) < 0.3).to(device)
    mask[..., 0] = True
    _check(ops.tree_attention(q, k, v, mask, scale), _reference(q, k, v, mask, scale))


def test_mfma_and_loop_kernels_agree(device):
    """The verification shape through the MFMA kernel (16-byte aligned rows)
    and through the loop kernel (a query view one element off alignment):
    both within the fp32 reference's tolerance, and within bf16 rounding of
    each other."""
    g = torch.Generator().manual_seed(12)
    tree = synthetic_tree(60, 6, seed=6, vocab=151936)
    base, Q, Hq, Hkv, D = 1024, 61, 32, 4, 128
    S = base + Q
    qbuf = _rand((1, Q, Hq, D + 8), device, g)
    q_aligned = qbuf[..., :D].transpose(1, 2)
    q_shifted = torch.empty((1, Q, Hq, D + 1), dtype=torch.bfloat16, device=device)
    q_shifted[..., 1:] = qbuf[..., :D]
    q_off = q_shifted[..., 1:].transpose(1, 2)  # same values, rows 2 bytes off alignment
    k = _rand((1, Hkv, S, D), device, g)
    v = _rand((1, Hkv, S, D), device, g)
    mask = tree.verification_attention_mask(base_kv_length=base, device=device)
    scale = D ** -0.5
    ref = _reference(q_aligned, k, v, mask, scale)
    fast = ops.tree_attention(q_aligned, k, v, mask, scale)
    loop = ops.tree_attention(q_off, k, v, mask, scale)
    _check(fast, ref)
    _check(loop, ref)
    assert ((fast.float() - loop.float()).abs().max() / ref.abs().max()).item() <= 1e-2


# Edges of the tiled form: 64-key tiles and 32- / 128-row tiles with remainders,
# keys fewer than queries (rows without a key give 0), one to many key splits,
# both forms with and without a mask, negative scales.
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 4, 128), (8, 4, 64), (16, 1, 64)])
@pytest.mark.parametrize("Q,S,scale", [(1, 63, 0.09), (1, 65, -0.09), (1, 4097, 0.09), (3, 2, 0.09),
                                       (17, 129, 0.1), (33, 1500, -0.1), (70, 64, 0.09),
                                       (129, 3000, 0.09), (300, 300, 0.09)])
def test_tiled_edges(device, Hq, Hkv, D, Q, S, scale):
    g = torch.Generator().manual_seed(Q * 7 + S + D)
    q = _rand((2, Q, Hq, D + 8), device, g)[..., :D].transpose(1, 2)  # padded token rows
    k = _rand((2, S, Hkv, D), device, g).transpose(1, 2)
    v = _rand((2, Hkv, S, D + 16), device, g)[..., :D]
    ref = _reference(q, k, v, None, scale)
    _check(ops.tree_attention(q, k, v, None, scale), ref)
    mask = (torch.rand((2, 1, Q, S + 3), generator=g) < 0.4).to(device)[..., 1:S + 1]
    mask[..., S // 2] = True
    out = ops.tree_attention(q, k, v, mask, scale)
    _check(out, _reference(q, k, v, mask, scale))
    assert torch.equal(out, ops.tree_attention(q, k, v, mask, scale))


def test_split_and_unsplit_calls_agree(device):
    """A call without scratch memory runs its keys in one split: the same
    values up to the order of the fp32 sums and the rounding of P, which is
    relative to the form's running maximum (_check's bounds)."""
    from specfit_amd import _native

    g = torch.Generator().manual_seed(31)
    Hq, Hkv, D, Q, S = 32, 4, 128, 2, 3001
    q, k, v = (_rand(s, device, g) for s in ((Hq, Q, D), (Hkv, S, D), (Hkv, S, D)))
    assert _native.lib().sf_tree_attention_workspace(Q, S, Hq, Hkv, D, 0) > 0
    split = ops.tree_attention(q[None], k[None], v[None], None, 0.09)[0]
    whole = torch.empty((Q, Hq, D), dtype=torch.bfloat16, device=device)
    rc = _native.lib().sf_tree_attention(
        q.data_ptr(), D, Q * D, k.data_ptr(), S * D, D, v.data_ptr(), S * D, D, None, 0, Q, S, Hq,
        Hkv, D, 0.09, whole.data_ptr(), torch.cuda.current_stream(device).cuda_stream)
    _native.check(rc, "sf_tree_attention")
    _check(split[None], whole[None].float())


def test_fully_masked_row_is_zero_and_large_logits_are_stable(device):
    g = torch.Generator().manual_seed(2)
    q = _rand((1, 8, 5, 128), device, g, std=30.0)
    k = _rand((1, 2, 200, 128), device, g, std=30.0)
    v = _rand((1, 2, 200, 128), device, g)
    mask = torch.ones((1, 1, 5, 200), dtype=torch.bool, device=device)
    mask[0, 0, 3] = False
    out = ops.tree_attention(q, k, v, mask, 0.088)
    assert torch.count_nonzero(out[0, 3]) == 0
    ref = _reference(q, k, v, mask, 0.088)
    keep = [0, 1, 2, 4]
    _check(out[:, keep], ref[:, keep])
    assert torch.isfinite(out.float()).all()


# Scores past 2^24, where a rounded product of the row maximum is off by more
# than the spacing of the exponents: both tile forms, masked and not, one and
# many key splits.
@pytest.mark.parametrize("std", [3e4, 1e5, 3e5, 1e15])
@pytest.mark.parametrize("Q,S,masked", [(1, 4096, False), (61, 1085, True), (40, 100, True),
                                        (200, 200, False), (1024, 1024, False),
                                        (700, 900, True)])
def test_large_finite_scores(device, Q, S, masked, std):
    """At these scales one key takes all of a row's weight, so the row is that
    key's values, bit for bit.  Rows whose two largest scores are closer than
    the error of an fp32 dot product of 128 terms (2^-24 * 128 of the sum of
    magnitudes, taken twice) are left out."""
    Hq, Hkv, D, scale = 16, 2, 128, 128 ** -0.5
    g = torch.Generator().manual_seed(Q + S)
    q, k = _rand((Hq, Q, D), device, g, std), _rand((Hkv, S, D), device, g, std)
    v = _rand((Hkv, S, D), device, g)
    allowed = torch.arange(S, device=device)[None] <= S - Q + torch.arange(Q, device=device)[:, None]
    mask = None
    if masked:
        allowed = (torch.rand((Q, S), generator=g) < 0.5).to(device)
        allowed[:, 0] = True
        mask = allowed[None, None].contiguous()
    for sign in (1.0, -1.0):
        out = ops.tree_attention(q[None], k[None], v[None], mask, sign * scale)[0]
        decided = 0
        for head in range(Hq):
            kd = k[head * Hkv // Hq].double()
            s = (sign * (q[head].double() @ kd.T)).masked_fill(~allowed, -math.inf)
            size = (q[head].double().abs() @ kd.abs().T).amax(-1)
            top = torch.cat([s, torch.full_like(s[:, :1], -math.inf)], dim=1).topk(2, dim=-1)
            gap = top.values[:, 0] - top.values[:, 1]
            rows = gap > 2 * 2 ** -24 * 128 * size + 200 / scale
            decided += int(rows.sum())
            want = v[head * Hkv // Hq][top.indices[:, 0]]
            assert torch.equal(out[rows, head], want[rows]), (head, sign)
        assert decided >= 0.9 * Q * Hq


@pytest.mark.parametrize("Q,S,masked", [(1, 4097, False), (61, 1085, True), (700, 700, False),
                                        (512, 3512, False), (2048, 2048, False)])
def test_rounding_of_the_probabilities(device, Q, S, masked):
    """The kernel's squared error against 64 bits, less that of rounding the
    result, is at most 0.85 of what rounding every probability to bf16 once
    gives: a quarter of the tiles carries the rounded-off rest too (and each
    wavefront's first), which leaves 0.75 of it at most, plus the scatter of
    these samples (about 3%) on either side."""
    Hq, Hkv, D = 16, 2, 128
    g = torch.Generator().manual_seed(Q)
    q, k, v = (_rand((h, n, D), device, g) for h, n in ((Hq, Q), (Hkv, S), (Hkv, S)))
    scale = D ** -0.5
    allowed = torch.arange(S, device=device)[None] <= S - Q + torch.arange(Q, device=device)[:, None]
    mask = allowed[None, None].contiguous() if masked else None
    out = ops.tree_attention(q[None], k[None], v[None], mask, scale)[0]
    err = result = once = 0.0
    for head in range(Hq):
        kd, vd = k[head * Hkv // Hq].double(), v[head * Hkv // Hq].double()
        s = (q[head].double() @ kd.T * scale).masked_fill(~allowed, -math.inf)
        p = torch.exp(s - s.amax(-1, keepdim=True))
        total = p.sum(-1, keepdim=True)
        want = p @ vd / total
        rounded = p.to(torch.bfloat16).double() @ vd / total
        err += (out[:, head].double() - want).square().sum().item()
        result += (want.to(torch.bfloat16).double() - want).square().sum().item()
        once += (rounded - want).square().sum().item()
    assert err - result <= 0.85 * once, (err - result) / once


def test_mask_without_heads_is_refused(device):
    """An empty head dimension holds no mask row; its null address must not
    become the causal rule."""
    q = torch.zeros((1, 4, 2, 64), dtype=torch.bfloat16, device=device)
    k = torch.zeros((1, 2, 5, 64), dtype=torch.bfloat16, device=device)
    for heads in (0, 4):
        mask = torch.zeros((1, heads, 2, 5), dtype=torch.bool, device=device)
        if heads:
            assert not ops.tree_attention(q, k, k, mask, 1.0).any()  # head 0 serves every head
        else:
            with pytest.raises(ValueError, match="mask"):
                ops.tree_attention(q, k, k, mask, 1.0)


def test_scratch_of_a_side_stream_call_is_the_side_streams(device):
    """A block that the current stream gave back, with a copy from it still
    queued there, is not the scratch of a call on another stream.  (The
    output is the current stream's memory: nothing small is given back here
    while it is in use.)"""
    from specfit_amd import _native

    g = torch.Generator().manual_seed(6)
    q, k, v = (_rand((1, h, n, 128), device, g) for h, n in ((32, 1), (4, 4096), (4, 4096)))
    ref = _reference(q, k, v, None, 0.09)
    need = _native.lib().sf_tree_attention_workspace(1, 4096, 32, 4, 128, 0)
    side, busy = torch.cuda.Stream(device), torch.randn(4096, 4096, device=device)
    result = torch.empty_like(busy)
    torch.cuda.synchronize()
    block = torch.full((need,), 7, dtype=torch.uint8, device=device)
    torch.cuda.synchronize()
    for _ in range(20):  # several ms of work before the copy
        torch.mm(busy, busy, out=result)
    copy = block.clone()
    del block
    outs = [ops.tree_attention(q, k, v, None, 0.09, stream=side) for _ in range(3)]
    torch.cuda.synchronize()
    assert bool((copy == 7).all())
    for out in outs:
        _check(out, ref)


def test_call_without_room_for_scratch_runs_unsplit(device, monkeypatch):
    g = torch.Generator().manual_seed(5)
    q, k, v = (_rand((1, h, n, 128), device, g) for h, n in ((32, 1), (4, 4096), (4, 4096)))
    ref = _reference(q, k, v, None, 0.09)
    empty, refused = torch.empty, []

    def full(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            refused.append(args)
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", full)
    out = ops.tree_attention(q, k, v, None, 0.09)
    monkeypatch.undo()
    assert refused
    _check(out, ref)


def test_call_without_scratch_uses_the_best_unsplit_form(device):
    """One token over 4096 keys without scratch: four key groups in a
    workgroup, about 5 times the split call's device time (9 us); one key
    group takes 9 times."""
    from specfit_amd import _native

    lib, stream = _native.lib(), torch.cuda.current_stream(device).cuda_stream
    Hq, Hkv, D, S = 32, 4, 128, 4096
    q, k, v, out = (torch.randn(s, device=device).to(torch.bfloat16)
                    for s in ((1, Hq, D), (Hkv, S, D), (Hkv, S, D), (1, Hq, D)))
    need = lib.sf_tree_attention_workspace(1, S, Hq, Hkv, D, 0)
    work = torch.empty(need, dtype=torch.uint8, device=device)

    def seconds(work_ptr, nbytes):
        times = []
        for _ in range(7):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(50):
                _native.check(lib.sf_tree_attention_split(
                    q.data_ptr(), Hq * D, D, k.data_ptr(), S * D, D, v.data_ptr(), S * D, D, None,
                    0, 1, S, Hq, Hkv, D, 0.09, out.data_ptr(), work_ptr, nbytes, stream), "split")
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[3]

    split, whole = seconds(work.data_ptr(), need), seconds(None, 0)
    assert whole < 7 * split, (whole, split)


@pytest.mark.parametrize("Q,S", [(61, 1085), (1024, 1024)])
def test_a_row_does_not_depend_on_the_scores_of_others(device, Q, S):
    Hq, Hkv, D = 8, 2, 128
    g = torch.Generator().manual_seed(Q)
    q, k, v = (_rand((1, h, n, D), device, g) for h, n in ((Hq, Q), (Hkv, S), (Hkv, S)))
    plain = ops.tree_attention(q, k, v, None, 0.09)
    q[0, ::2, ::3] *= 1e6
    mixed = ops.tree_attention(q, k, v, None, 0.09)
    rows = torch.ones((Q, Hq), dtype=torch.bool, device=device)
    rows[::3, ::2] = False
    assert torch.equal(mixed[0][rows], plain[0][rows])


@pytest.mark.parametrize("Q,S,masked", [(1, 4096, False), (61, 1085, True), (200, 200, False),
                                        (1024, 1024, False), (700, 900, True), (5, 1056, False)])
def test_infinities_and_nan(device, Q, S, masked):
    """An infinite value stays infinite for the rows that admit its key; NaN
    and infinite scores touch their own rows only (zeros, as in the loop form,
    whose sum is NaN there too)."""
    Hq, Hkv, D = 8, 2, 128
    g = torch.Generator().manual_seed(Q)
    q, k, v = (_rand((1, h, n, D), device, g) for h, n in ((Hq, Q), (Hkv, S), (Hkv, S)))
    mask = torch.ones((1, 1, Q, S), dtype=torch.bool, device=device) if masked else None
    clean = ops.tree_attention(q, k, v, mask, 0.09)
    for key in (0, 63, S // 2, S - Q, S - 1):
        for value in (math.inf, -math.inf):
            bad = v.clone()
            bad[0, 1, key, 7] = value
            out = ops.tree_attention(q, k, bad, mask, 0.09)
            first = 0 if masked else max(0, key - (S - Q))  # rows that admit the key
            assert bool((out[0, first:, Hq // 2:, 7] == value).all()), (key, value)
            keep = torch.ones_like(out, dtype=torch.bool)
            keep[0, :, Hq // 2:, 7] = False  # equal but for the rest of P's rounding
            err = (out.float() - clean.float())[keep].abs().max()
            assert err.item() <= 1e-2 * clean.float().abs().max().item()
    for value in (math.nan, math.inf):
        bad = q.clone()
        bad[0, 3, Q // 2, 5] = value
        out = ops.tree_attention(bad, k, v, mask, 0.09)
        rows = torch.ones((Q, Hq), dtype=torch.bool, device=device)
        rows[Q // 2, 3] = False
        assert torch.equal(out[0][rows], clean[0][rows])
        assert not out[0, Q // 2, 3].any()
    # A key of -inf in one element: weight 0 for rows with a positive query
    # there (the row is that of the other keys), zeros for the others.
    bad = k.clone()
    bad[0, 0, S - Q, 9] = -math.inf
    out = ops.tree_attention(q, bad, v, mask, 0.09)
    without = torch.ones((1, 1, Q, S), dtype=torch.bool, device=device) if masked else (
        torch.arange(S, device=device) <= S - Q + torch.arange(Q, device=device)[:, None])[None, None]
    without = without.clone()
    without[..., S - Q] = False
    ref = _reference(q, k, v, without, 0.09)
    positive = (q[0, :Hq // 2, :, 9] > 0).T  # [Q, heads of KV head 0]
    got, want = out[0, :, :Hq // 2][positive], ref[0, :, :Hq // 2][positive]
    _check(got, want)
    negative = (q[0, :Hq // 2, :, 9] < 0).T
    assert not out[0, :, :Hq // 2][negative].any()


def test_argument_errors(device):
    q = torch.zeros((1, 4, 2, 8), dtype=torch.bfloat16, device=device)
    k = torch.zeros((1, 3, 5, 8), dtype=torch.bfloat16, device=device)
    with pytest.raises(ValueError, match="multiple"):
        ops.tree_attention(q, k, k, None, 1.0)
    k = torch.zeros((1, 2, 5, 8), dtype=torch.bfloat16, device=device)
    with pytest.raises(TypeError, match="bool"):
        ops.tree_attention(q, k, k, torch.zeros((1, 1, 2, 5), device=device), 1.0)
    with pytest.raises(ValueError, match="mask"):
        ops.tree_attention(q, k, k, torch.ones((1, 1, 2, 4), dtype=torch.bool, device=device), 1.0)


# ------------------------------------------------------------ model level --
def _tiny_model(layers=2, seed=7):
    from transformers import Qwen3MoeConfig, Qwen3MoeForCausalLM

    torch.manual_seed(seed)
    config = Qwen3MoeConfig(vocab_size=64, hidden_size=32, intermediate_size=48,
                            moe_intermediate_size=16, num_hidden_layers=layers,
                            num_attention_heads=4, num_key_value_heads=2, num_experts=4,
                            num_experts_per_tok=2, max_position_embeddings=64, bos_token_id=1,
                            eos_token_id=63, pad_token_id=62, norm_topk_prob=True)
    return Qwen3MoeForCausalLM(config).to(torch.bfloat16).eval()


def _offloaded(model, device, attn):
    register_tree_attention()
    model.config._attn_implementation = attn
    return build_offloaded_qwen3(model, device=device, slots_per_layer=2)


def _tree():
    return Eagle3DraftTree(
        token_ids=(5, 6, 9, 10), parent_ids=(0, 0, 1, 2), depths=(1, 1, 2, 2),
        conditional_probabilities=(0.6, 0.4, 0.5, 0.5),
        cumulative_log_probabilities=(math.log(0.6), math.log(0.4), math.log(0.6 * 0.5),
                                      math.log(0.4 * 0.5)))


@torch.inference_mode()
def test_each_tree_node_matches_an_independent_causal_path(device):
    loaded = _offloaded(_tiny_model(1), device, TREE_ATTENTION)
    target = loaded.model
    prefix = torch.tensor([[1, 7, 11]], device=device)
    tree = _tree()
    prefill = target(input_ids=prefix, attention_mask=torch.ones_like(prefix), use_cache=True,
                     logits_to_keep=1)
    seed = prefill.logits.argmax(dim=-1)
    verify_ids = tree.verification_token_ids(seed)
    tree_out = target(input_ids=verify_ids,
                      attention_mask=tree.verification_attention_mask(
                          base_kv_length=prefix.shape[1], device=device),
                      position_ids=tree.verification_position_ids(
                          base_kv_length=prefix.shape[1], device=device),
                      past_key_values=prefill.past_key_values, use_cache=True, logits_to_keep=0)
    for node in range(1 + tree.draft_node_count):
        path = []
        cur = node
        while cur:
            path.append(tree.token_ids[cur - 1])
            cur = tree.parent_ids[cur - 1]
        path.reverse()
        ids = torch.cat((prefix, seed, prefix.new_tensor(path).unsqueeze(0)), dim=1)
        expected = target(input_ids=ids, attention_mask=torch.ones_like(ids), use_cache=False,
                          logits_to_keep=1).logits[0, -1].float()
        actual = tree_out.logits[0, node].float()
        torch.testing.assert_close(actual, expected, atol=3e-2 * expected.abs().max().item(),
                                   rtol=3e-2)
        top2 = expected.topk(2).values
        if (top2[0] - top2[1]).item() > 0.05 * expected.abs().max().item():
            assert int(actual.argmax()) == int(expected.argmax())
    loaded.close()


@torch.inference_mode()
def test_tree_attention_model_matches_sdpa_model(device):
    base = _tiny_model(2, seed=9)
    state = {k: v.clone() for k, v in base.state_dict().items()}
    ours = _offloaded(base, device, TREE_ATTENTION)
    ref_model = _tiny_model(2, seed=9)
    ref_model.load_state_dict(state)
    theirs = _offloaded(ref_model, device, "sdpa")
    ids = torch.tensor([[1, 5, 9, 12, 3, 44, 21]], device=device)
    a = ours.model(input_ids=ids, attention_mask=torch.ones_like(ids)).logits.float()
    b = theirs.model(input_ids=ids, attention_mask=torch.ones_like(ids)).logits.float()
    torch.testing.assert_close(a, b, atol=3e-2 * b.abs().max().item(), rtol=3e-2)
    ours.close()
    theirs.close()


@torch.inference_mode()
def test_verify_draft_tree_commits_the_accepted_path(device):
    from transformers import DynamicCache

    loaded = _offloaded(_tiny_model(2, seed=4), device, TREE_ATTENTION)
    target = loaded.model
    prefix = torch.tensor([[1, 7, 11, 19]], device=device)
    cache = DynamicCache()
    prefill = target(input_ids=prefix, attention_mask=torch.ones_like(prefix),
                     past_key_values=cache, use_cache=True, logits_to_keep=1)
    seed = prefill.logits.argmax(dim=-1)
    # A chain that follows the target's own greedy decode is accepted whole
    # (up to bf16 near-ties), plus distractor siblings that never are.
    chain, ids = [], torch.cat((prefix, seed), dim=1)
    for _ in range(3):
        nxt = int(target(input_ids=ids, attention_mask=torch.ones_like(ids),
                         use_cache=False, logits_to_keep=1).logits[0, -1].argmax())
        chain.append(nxt)
        ids = torch.cat((ids, ids.new_tensor([[nxt]])), dim=1)
    tokens, parents, depths, probs = [], [], [], []
    parent = 0
    for depth, tok in enumerate(chain, start=1):
        tokens += [tok, (tok + 1) % 61]
        parents += [parent, parent]
        depths += [depth, depth]
        probs += [0.7, 0.3]
        parent = len(tokens) - 1
    cums, cum = [], {0: 0.0}
    for node, (p, par) in enumerate(zip(probs, parents), start=1):
        cum[node] = cum[par] + math.log(p)
        cums.append(cum[node])
    tree = Eagle3DraftTree(tuple(tokens), tuple(parents), tuple(depths), tuple(probs), tuple(cums))
    base = cache.get_seq_length()
    result = verify_draft_tree(target, tree, seed, cache)
    assert result.base_kv_length == base
    assert result.verification_positions == (0,) + result.accepted_node_ids
    assert cache.get_seq_length() == base + len(result.verification_positions)
    assert result.accepted_node_ids == tree.accepted_path(result.verifier_tokens)
    assert torch.equal(result.committed, result.verify_ids[:, result.verification_positions])
    last = result.verification_positions[-1]
    assert torch.equal(result.pending_seed, result.verifier_tokens[:, last:last + 1])
    # The seed's verification logits equal a causal forward of [prefix, seed].
    ids = torch.cat((prefix, seed), dim=1)
    expected = target(input_ids=ids, attention_mask=torch.ones_like(ids), use_cache=False,
                      logits_to_keep=1).logits[0, -1].float()
    torch.testing.assert_close(result.logits[0, 0].float(), expected,
                               atol=3e-2 * expected.abs().max().item(), rtol=3e-2)
    # The committed cache continues decoding: one more step runs on it.
    nxt = target(input_ids=result.pending_seed, past_key_values=cache, use_cache=True)
    assert cache.get_seq_length() == base + len(result.verification_positions) + 1
    assert torch.isfinite(nxt.logits.float()).all()
    loaded.close()
