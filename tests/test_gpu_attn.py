"""Variable-length causal GQA attention (torch.ops.talm.attn_fwd / attn_bwd / attn_bwd_rope)
against per-row causal SDPA in fp32 on the CPU (solution/unpad.py:121-134): output, log-sum-exp
and the gradients of q, k, v. fp16 operands, fp32 statistics, fp16 P and dS in the MFMA products: the
tolerances are stated per tensor relative to its largest reference magnitude."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

HQ, HKV, D = 12, 2, 128


def _reference(q, k, v, lengths, scale, dout):
    """fp32 CPU: per sequence, causal softmax(scale q k^T) v with KV heads shared by groups of
    query heads; returns out, lse [Hq, N] and (dq, dk, dv) for the upstream gradient dout."""
    q, k, v = (t.detach().float().cpu().requires_grad_(True) for t in (q, k, v))
    outs, lses = [], []
    s0 = 0
    group = q.shape[1] // k.shape[1]
    for n in lengths:
        qs = q[s0:s0 + n].transpose(0, 1)                                  # [Hq, n, D]
        ks = k[s0:s0 + n].transpose(0, 1).repeat_interleave(group, 0)      # [Hq, n, D]
        vs = v[s0:s0 + n].transpose(0, 1).repeat_interleave(group, 0)
        scores = scale * qs @ ks.transpose(1, 2)
        mask = torch.ones(n, n, dtype=torch.bool).triu(1)
        scores = scores.masked_fill(mask, float("-inf"))
        lses.append(torch.logsumexp(scores, -1))                           # [Hq, n]
        outs.append((torch.softmax(scores, -1) @ vs).transpose(0, 1))     # [n, Hq, D]
        s0 += n
    out = torch.cat(outs)
    out.backward(dout.float().cpu())
    return out.detach(), torch.cat(lses, 1).detach(), q.grad, k.grad, v.grad


def _close(name, got, ref, rel):
    got = got.float().cpu()
    scale = ref.abs().max().item()
    err = (got - ref).abs().max().item()
    print(f"[attn] {name}: max err {err:.3e} (max |ref| {scale:.3e})", flush=True)
    assert err <= rel * scale + 1e-6, f"{name}: max error {err} > {rel} x {scale}"


def _run(lengths, strided, seed, HQ=HQ, HKV=HKV):
    import talm_amd._ops  # noqa: F401
    from talm_amd import _ops

    g = torch.Generator("cpu").manual_seed(seed)
    n = sum(lengths)
    if strided:  # the q|k|v node's layout: q and k column views of one [N, 2048] buffer
        qkv = torch.randn(n, (HQ + HKV) * D, generator=g).half().cuda()
        q = qkv[:, :HQ * D].view(n, HQ, D)
        k = qkv[:, HQ * D:].view(n, HKV, D)
    else:
        q = torch.randn(n, HQ, D, generator=g).half().cuda()
        k = torch.randn(n, HKV, D, generator=g).half().cuda()
    v = torch.randn(n, HKV, D, generator=g).half().cuda()
    dout = torch.randn(n, HQ, D, generator=g).half().cuda()
    cu = torch.tensor([0] + list(torch.tensor(lengths).cumsum(0)), dtype=torch.int32).cuda()
    scale = 1.0 / math.sqrt(D)
    out = torch.empty(n, HQ, D, dtype=torch.float16, device="cuda")
    lse = torch.empty(HQ, n, dtype=torch.float32, device="cuda")
    torch.ops.talm.attn_fwd(q, k, v, cu, max(lengths), scale, out, lse)
    dq = torch.empty_like(out)
    dk = torch.empty(n, HKV, D, dtype=torch.float16, device="cuda")
    dv = torch.empty_like(dk)
    ws = torch.empty(_ops.attn_bwd_workspace_bytes(n, HQ), dtype=torch.uint8, device="cuda")
    torch.ops.talm.attn_bwd(q, k, v, out, dout, lse, cu, max(lengths), scale, dq, dk, dv, ws)
    torch.cuda.synchronize()
    r_out, r_lse, r_dq, r_dk, r_dv = _reference(q, k, v, lengths, scale, dout)
    _close("out", out, r_out, 2e-3)
    _close("lse", lse, r_lse, 1e-4)
    _close("dq", dq, r_dq, 4e-3)
    _close("dk", dk, r_dk, 4e-3)
    _close("dv", dv, r_dv, 4e-3)


@pytest.mark.parametrize("lengths,strided,seed", [
    ([300, 128, 512, 257], True, 1),    # config-5-like packed batch, the q|k|v buffer's views
    ([1, 17, 64, 65, 129], False, 2),   # single-token and tile-boundary sequences
    ([512], False, 3),
])
def test_attention_matches_per_row_causal_sdpa(lengths, strided, seed):
    print(f"[case] attention lengths={lengths} strided={strided} seed={seed}", flush=True)
    _run(lengths, strided, seed)


@pytest.mark.parametrize("lengths,hq,hkv,seed", [
    ([1, 2000, 64, 65, 700, 1500, 1, 1111], 12, 2, 21),   # one grid axis, 64-row tiles, mixed lengths
    ([1024, 33, 128, 129, 900, 1, 800, 1900], 16, 16, 22),      # 128-row tiles
    ([300] + [9 * i % 250 + 1 for i in range(63)], 16, 4, 23),  # 64 sequences, 32-row tiles
])
def test_attention_listed_longest_first(lengths, hq, hkv, seed):
    """More workgroups than a round over sequences of different length: taken from the list."""
    print(f"[case] attention listed seqs={len(lengths)} heads={hq}/{hkv} seed={seed}", flush=True)
    _run(lengths, False, seed, hq, hkv)


@pytest.mark.parametrize("lengths,hq,hkv,seed", [
    ([2048, 31], 12, 2, 11),       # few workgroups, a long chain: the key tiles split in two
    ([449, 64, 1], 4, 1, 12),      # four heads per workgroup, split (8 key tiles), one-tile rows
    ([448, 33], 4, 1, 13),         # the same below the split's chain length
    ([130, 127, 128, 129], 7, 1, 14),    # one head per workgroup: 128-row tiles and their edges
    ([320] * 24, 16, 8, 15),       # more workgroups than two rounds: unsplit, group of 2
    ([1100, 65], 8, 8, 16),        # no grouping, split
])
def test_attention_over_head_groups_and_key_splits(lengths, hq, hkv, seed):
    """Every (heads per workgroup, key split) form of the forward, at its tile edges."""
    print(f"[case] attention lengths={lengths} heads={hq}/{hkv} seed={seed}", flush=True)
    _run(lengths, True, seed, hq, hkv)


@pytest.mark.parametrize("lengths,hq,hkv", [
    ([16, 1, 31, 32], 12, 4), ([33, 64, 0, 63], 9, 1),  # three heads a workgroup: up to 64 rows
    ([65, 16], 12, 4),                                  # one head a workgroup
    ([40, 64], 6, 1),                                   # two
])
def test_attention_of_short_rows_in_groups_of_three(lengths, hq, hkv):
    """Workgroups of three heads with a fourth wavefront that has none, against the same reference."""
    print(f"[case] attention short rows {lengths} heads={hq}/{hkv}", flush=True)
    _run(lengths, True, 31, hq, hkv)


@pytest.mark.parametrize("n,pos", [(256, 64), (256, 200), (600, 70), (600, 255)])
def test_attention_largest_weight_of_the_first_tiles_is_exact(n, pos):
    """Every score is 0 except key `pos`'s 5 (7.2 in log2 units, below the lazy rescale), and v is 0
    except at that key: out = v e^5 / (e^5 + i). With the key's weight held as 1 its product is
    exact, and what remains is the fp16 rounding of the output (2^-11) and that of an fp32 sum of n
    terms; as e^5 relative to an earlier reference it adds fp16's error of 148.41, 2.6e-4."""
    import talm_amd._ops  # noqa: F401

    g = torch.Generator("cpu").manual_seed(n + pos)
    q, k, v = torch.zeros(n, 1, D), torch.zeros(n, 1, D), torch.zeros(n, 1, D)
    q[:, 0, 0] = 1.0
    k[pos, 0, 0] = 5.0
    v[pos, 0] = (1 + torch.rand(D, generator=g)).half().float()
    cu = torch.tensor([0, n], dtype=torch.int32).cuda()
    out = torch.empty(n, 1, D, dtype=torch.float16, device="cuda")
    lse = torch.empty(1, n, dtype=torch.float32, device="cuda")
    torch.ops.talm.attn_fwd(q.half().cuda(), k.half().cuda(), v.half().cuda(), cu, n, 1.0, out, lse)
    rows = torch.arange(pos, n, dtype=torch.float64)
    ref = v[pos, 0].double() * (math.exp(5) / (math.exp(5) + rows))[:, None]
    err = ((out[pos:, 0].double().cpu() - ref) / ref).abs().max().item()
    print(f"[attn] relative error {err:.3e}", flush=True)
    assert err <= 2.0 ** -11 + n * 2.0 ** -24
    assert not out[:pos].any()


def _rotate_back(dy, cos, sin):
    """The gradient of x -> x cos + rotate_half(x) sin (transformers' apply_rotary_pos_emb on one
    [N, H, 128] tensor, fp32 CPU) at dy, by autograd: the rotary backward the fused kernel folds
    in, derived from the forward rather than restated."""
    x = torch.zeros_like(dy, requires_grad=True)
    half = x.shape[-1] // 2
    rotated = torch.cat((-x[..., half:], x[..., :half]), -1)
    (x * cos[:, None, :] + rotated * sin[:, None, :]).backward(dy)
    return x.grad


@pytest.mark.parametrize("lengths,seed", [
    ([300, 128, 512, 257], 4),          # config-5-like packed batch
    ([1, 17, 64, 65, 129], 5),          # single-token and tile-boundary sequences
])
def test_attention_backward_with_the_rotary_backward_folded_in(lengths, seed):
    """attn_bwd_rope: dq / dk rotated back in the kernel's epilogues equal the reference's
    attention gradients pushed through the rotary embedding's backward. cos / sin are independent
    random rows (not the model's tables, whose two halves are equal) so that a swapped half or
    a cos read in place of a sin fails, and their rows are strided (160 of which 128 are read).
    The outputs are column views of one [N, q + k + v] buffer, as in the attention block."""
    import talm_amd._ops  # noqa: F401
    from talm_amd import _ops

    print(f"[case] attention+rope backward lengths={lengths} seed={seed}", flush=True)
    g = torch.Generator("cpu").manual_seed(seed)
    n = sum(lengths)
    qkv = torch.randn(n, (HQ + 2 * HKV) * D, generator=g).half().cuda()
    q = qkv[:, :HQ * D].view(n, HQ, D)
    k = qkv[:, HQ * D:(HQ + HKV) * D].view(n, HKV, D)
    v = qkv[:, (HQ + HKV) * D:].view(n, HKV, D)
    dout = torch.randn(n, HQ, D, generator=g).half().cuda()
    cs = torch.rand(2, n, 160, generator=g) * 2 - 1
    cos, sin = cs[0].cuda()[:, :D], cs[1].cuda()[:, :D]
    cu = torch.tensor([0] + list(torch.tensor(lengths).cumsum(0)), dtype=torch.int32).cuda()
    scale = 1.0 / math.sqrt(D)
    out = torch.empty(n, HQ, D, dtype=torch.float16, device="cuda")
    lse = torch.empty(HQ, n, dtype=torch.float32, device="cuda")
    torch.ops.talm.attn_fwd(q, k, v, cu, max(lengths), scale, out, lse)
    grads = torch.full_like(qkv, float("nan"))
    dq = grads[:, :HQ * D].view(n, HQ, D)
    dk = grads[:, HQ * D:(HQ + HKV) * D].view(n, HKV, D)
    dv = grads[:, (HQ + HKV) * D:].view(n, HKV, D)
    ws = torch.empty(_ops.attn_bwd_workspace_bytes(n, HQ), dtype=torch.uint8, device="cuda")
    torch.ops.talm.attn_bwd_rope(q, k, v, out, dout, lse, cu, max(lengths), scale, cos, sin, dq,
                                 dk, dv, ws)
    torch.cuda.synchronize()
    _r_out, _r_lse, r_dq, r_dk, r_dv = _reference(q, k, v, lengths, scale, dout)
    c, s_ = cos.cpu(), sin.cpu()
    assert not grads.isnan().any(), "a gradient element was not written"
    _close("dq (rotated back)", dq, _rotate_back(r_dq, c, s_), 4e-3)
    _close("dk (rotated back)", dk, _rotate_back(r_dk, c, s_), 4e-3)
    _close("dv", dv, r_dv, 4e-3)


@pytest.mark.parametrize("lengths,hq,hkv", [
    ([0, 1, 128, 129, 700, 1500, 0, 333], 12, 2),      # empty sequences, tile edges
    ([7 * i % 300 for i in range(64)], 12, 2),         # one sequence per lane
    ([7 * i % 300 for i in range(65)], 12, 2),         # one more: no queue
    ([2305], 16, 8),                                   # 608 items: just above two per CU of 256
    ([96] * 31 + [97], 12, 2),                         # one tile each, 96 rows on the average or more
    ([96] * 32, 12, 2),                                # not more: no queue
])
def test_attention_backward_from_the_queue(lengths, hq, hkv):
    """The same workgroups' work whether drawn from the queue or launched one by one (a workspace
    without the queue's counter): the same bits, every element written, twice in a row."""
    import talm_amd._ops  # noqa: F401
    from talm_amd import _ops

    print(f"[case] attention queue seqs={len(lengths)} heads={hq}/{hkv}", flush=True)
    n = sum(lengths)
    g = torch.Generator().manual_seed(n)
    q, dout = (torch.randn(n, hq, D, generator=g).half().cuda() for _ in range(2))
    k, v = (torch.randn(n, hkv, D, generator=g).half().cuda() for _ in range(2))
    cu = torch.tensor([0] + lengths).cumsum(0).to("cuda", torch.int32)
    out = torch.empty_like(q)
    lse = torch.empty(hq, n, dtype=torch.float32, device="cuda")
    torch.ops.talm.attn_fwd(q, k, v, cu, max(lengths), D ** -0.5, out, lse)
    size = _ops.attn_bwd_workspace_bytes(n, hq)
    runs = []
    for nbytes in (size - 256, size, size):
        ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device="cuda")
        grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        torch.ops.talm.attn_bwd(q, k, v, out, dout, lse, cu, max(lengths), D ** -0.5, *grads, ws)
        runs.append(grads)
    for grads in runs:
        for got, ref in zip(grads, runs[0]):
            assert not got.isnan().any() and torch.equal(got, ref)


def test_attention_rope_backward_rejects_bad_tables():
    import talm_amd._ops  # noqa: F401
    from talm_amd import _ops

    n = 8
    q = torch.zeros(n, HQ, D, dtype=torch.float16, device="cuda")
    k = torch.zeros(n, HKV, D, dtype=torch.float16, device="cuda")
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    lse = torch.zeros(HQ, n, device="cuda")
    ws = torch.empty(_ops.attn_bwd_workspace_bytes(n, HQ), dtype=torch.uint8, device="cuda")
    narrow = torch.zeros(n, 64, device="cuda")                    # fewer than 128 columns
    with pytest.raises(ValueError):
        torch.ops.talm.attn_bwd_rope(q, k, k, q, q, lse, cu, n, 0.125, narrow, narrow, q, k, k, ws)
    odd = torch.zeros(n, 131, device="cuda")[:, :128]             # row stride not a multiple of 4
    with pytest.raises(ValueError):
        torch.ops.talm.attn_bwd_rope(q, k, k, q, q, lse, cu, n, 0.125, odd, odd, q, k, k, ws)


def test_attention_rejects_bad_shapes():
    import talm_amd._ops  # noqa: F401

    n = 8
    q = torch.zeros(n, HQ, 64, dtype=torch.float16, device="cuda")  # head_dim 64: not supported
    k = torch.zeros(n, HKV, 64, dtype=torch.float16, device="cuda")
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        torch.ops.talm.attn_fwd(q, k, k, cu, n, 0.125, q, torch.empty(HQ, n, device="cuda"))
