"""Parity of the fused LM head + cross-entropy (talm_head_ce, MFMA) with the CPU oracle.

Bars (the reference's own head tests solution/test_kernels.py:134-184 and
fuzz bounds solution/test_fuzz.py:293-331):
- per-token loss / entropy: |ours - ref| <= 2e-5 + 2e-6 * max|z| (loss) and 2e-5 + 1e-5 * max|z|
  (entropy) on exact-style inputs; 1e-4 relative on the mean loss;
- argmax / correctness: bit-exact on exact-style inputs (every logit exact in fp16), and on
  Gaussian inputs everywhere except rows with a near tie ("fragile", :175-176);
- dH: rtol 2e-3, atol 2^-7 * max|dH| (solution/test_kernels.py:182-184).
"""

import numpy as np
import pytest
import torch

from oracle import head as head_oracle
from talm_amd import _ops, fused_head, workloads
from tests.test_oracle import exact_head_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(msg):
    print(f"[case] {msg}", flush=True)


def _run(h16, w16, t, num_items=None, vchunk=8192, grad_scale=3.0, grad_all_rows=False):
    x = torch.from_numpy(h16).to(DEV).requires_grad_()
    w = torch.from_numpy(w16).to(DEV)
    tt = torch.from_numpy(t).to(DEV)
    loss, tl, ent, corr, arg = fused_head.fused_head_loss(x, w, tt, num_items, vchunk,
                                                          return_argmax=True,
                                                          grad_all_rows=grad_all_rows)
    (loss * grad_scale).backward()
    return {"loss": float(loss.detach()), "token_loss": tl.cpu().numpy(), "entropy": ent.cpu().numpy(),
            "correct": corr.cpu().numpy(), "best_idx": arg.cpu().numpy(),
            "grad": x.grad.float().cpu().numpy()}


def _check(res, h16, w16, t, vchunk, num_items=None, grad_scale=3.0, exact=True, what=""):
    ref = head_oracle.head_direct(h16, w16, t)
    zmax = ref["zmax"]
    tol_loss = 2e-5 + 2e-6 * zmax
    tol_ent = 2e-5 + 1e-5 * zmax
    if not exact:
        tol_loss = tol_loss + 8 * 2.0 ** -11 * zmax
        tol_ent = tol_ent + 16 * 2.0 ** -11 * zmax
    assert np.all(np.abs(res["token_loss"] - ref["token_loss"]) <= tol_loss), f"{what}: loss"
    assert np.all(np.abs(res["entropy"] - ref["entropy"]) <= tol_ent), f"{what}: entropy"
    lab = t >= 0
    assert np.all(res["token_loss"][~lab] == 0), f"{what}: loss on unlabelled rows"
    if exact:
        assert np.array_equal(res["best_idx"], ref["best_idx"]), f"{what}: argmax"
        assert np.array_equal(res["correct"], ref["correct"]), f"{what}: correct"
    loss_ref, denom = head_oracle.loss(ref["token_loss"], t, num_items)
    assert abs(res["loss"] - loss_ref) <= 1e-4 * abs(loss_ref) + 1e-6, f"{what}: mean loss"
    g_ref = ref["grad"] * grad_scale / denom
    scale = np.abs(g_ref).max() if g_ref.size else 0.0
    assert np.all(np.abs(res["grad"] - g_ref) <= 2e-3 * np.abs(g_ref) + 2.0 ** -7 * scale), \
        f"{what}: dH"
    assert np.all(res["grad"][~lab] == 0), f"{what}: gradient on unlabelled rows"
    return ref


def _head_ce_by_group(h, w, t, vchunk, n_grad, group):
    """talm_head_ce with a workspace that holds `group` slices a step and no more (for inputs
    where a step would take more): as fused_head.head_ce returns it."""
    n, hidden = h.shape
    vocab = w.shape[0]
    size = _ops.head_ce_workspace_bytes(n, hidden, group * vchunk, vchunk, n_grad, group)
    assert size < _ops.head_ce_workspace_bytes(n, hidden, vocab, vchunk, n_grad, group)
    out = {k: torch.empty(n, dtype=d, device=DEV) for k, d in
           (("token_loss", torch.float32), ("entropy", torch.float32),
            ("best_idx", torch.int32), ("correct", torch.int32))}
    out["grad"] = torch.empty_like(h) if n_grad else None
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    torch.ops.talm.head_ce(h, w, t, vchunk, n_grad, group, *out.values(), ws)
    return out


@pytest.mark.parametrize("n,hidden,vocab,vchunk,seed", [
    (37, 64, 4097, 4096, 1), (300, 256, 1000, 384, 2), (5, 1536, 151936, 8192, 3),
    (2, 16, 5, 128, 4), (129, 32, 20000, 8192, 5), (64, 8, 1, 128, 6)])
def test_head_exact_style_matches_oracle(n, hidden, vocab, vchunk, seed):
    """Exact-style inputs (every logit exact in fp16: solution/test_fuzz.py:225-256): argmax and
    correctness bit-exact, statistics to fp32 rounding, dH to the reference's bound; also
    checked against the oracle's own online restatement at the same slice width."""
    _case(f"head exact n={n} H={hidden} V={vocab} vchunk={vchunk}")
    h16, w16, t = exact_head_case(n, hidden, vocab, seed)
    res = _run(h16, w16, t, vchunk=vchunk)
    _check(res, h16, w16, t, vchunk, what="direct")
    online = head_oracle.head_ce(h16, w16, t, vchunk=vchunk)
    assert np.array_equal(res["best_idx"], online["best_idx"])
    np.testing.assert_allclose(res["token_loss"], online["token_loss"], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("labels", ["none", "all", "one"])
def test_head_label_edge_cases(labels):
    _case(f"head labels={labels}")
    h16, w16, t = exact_head_case(70, 64, 3000, 7)
    if labels == "none":
        t[:] = -100
    elif labels == "all":
        t = np.random.default_rng(8).integers(0, 3000, 70)
    else:
        t[:] = -100
        t[33] = 1234
    res = _run(h16, w16, t, vchunk=1024)
    _check(res, h16, w16, t, 1024, what=labels)


@pytest.mark.parametrize("labels", ["mixed", "none", "one", "all"])
def test_head_every_row_a_gradient_row(labels):
    """grad_all_rows (the fixed-shape step captured in a HIP graph): no labelled-first
    reordering, every row goes through the gradient GEMM; an ignored row's gradient is exactly
    zero and the rest matches the oracle to the same bars."""
    _case(f"head every row a gradient row, labels={labels}")
    h16, w16, t = exact_head_case(150, 64, 5000, 12)
    if labels == "none":
        t[:] = -100
    elif labels == "one":
        t[:] = -100
        t[77] = 4321
    elif labels == "all":
        t = np.random.default_rng(13).integers(0, 5000, 150)
    res = _run(h16, w16, t, vchunk=1024, grad_all_rows=True)
    _check(res, h16, w16, t, 1024, what=f"all rows {labels}")


@pytest.mark.parametrize("stride", [0, 8])
def test_head_orders_overlapping_rows(stride):
    """Hidden rows that share memory (an expanded row, stride 0, or rows 8 columns apart) with
    some labels ignored: the same as of a contiguous copy, bit for bit."""
    _case(f"head overlapping rows, stride {stride}")
    h16, w16, t = exact_head_case(37, 64, 1000, 22)
    base = torch.from_numpy(h16).to(DEV).flatten()
    rows = base.as_strided((37, 64), (stride, 1))
    assert 0 < int((t >= 0).sum()) < 37
    outs = []
    for x in (rows.contiguous(), rows):
        x = x.detach().requires_grad_()
        loss, *per_row = fused_head.fused_head_loss(x, torch.from_numpy(w16).to(DEV),
                                                    torch.from_numpy(t).to(DEV), None, 256)
        loss.backward()
        outs.append([loss.detach(), *per_row, x.grad])
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("off", [-3, 2])
def test_head_wrong_label_count_is_not_silent(off):
    """A label count that is not the targets' own leaves rows without a place in the labelled-first
    order: the loss and those rows' outputs and gradients are NaN, the other rows' are right."""
    _case(f"head label count off by {off}")
    h16, w16, t = exact_head_case(300, 64, 1000, 23)
    count = int((t >= 0).sum())
    x = torch.from_numpy(h16).to(DEV).requires_grad_()
    w, tt = torch.from_numpy(w16).to(DEV), torch.from_numpy(t).to(DEV)
    ref = fused_head.fused_head_loss(x, w, tt, 1.0, 256, n_labelled=count, return_argmax=True)
    (ref_grad,) = torch.autograd.grad(ref[0], x)
    got = fused_head.fused_head_loss(x, w, tt, 1.0, 256, n_labelled=count + off, return_argmax=True)
    (grad,) = torch.autograd.grad(got[0], x)
    assert got[0].isnan()
    # the last labelled rows past the count, or the last unlabelled rows past the end
    lost = (tt >= 0).nonzero().flatten()[off:] if off < 0 else (tt < 0).nonzero().flatten()[-off:]
    kept = torch.ones(300, dtype=torch.bool, device=DEV)
    kept[lost] = False
    assert got[1][lost].isnan().all() and got[2][lost].isnan().all() and grad[lost].isnan().all()
    assert not got[3][lost].any() and (got[4][lost] == -1).all()
    for a, b in zip((*got[1:], grad), (*ref[1:], ref_grad)):
        assert torch.equal(a[kept], b[kept])


@pytest.mark.parametrize("num_items", [None, 7, "tensor"])
def test_head_num_items_denominator(num_items):
    _case(f"head num_items={num_items}")
    h16, w16, t = exact_head_case(40, 32, 900, 9)
    n_lab = int((t >= 0).sum())
    items = torch.tensor(n_lab + 3, device=DEV) if num_items == "tensor" else num_items
    ref_items = n_lab + 3 if num_items == "tensor" else num_items
    res = _run(h16, w16, t, num_items=items, vchunk=256)
    _check(res, h16, w16, t, 256, num_items=ref_items)


def test_head_argmax_ties_across_slices_and_groups():
    """solution/test_kernels.py:250-282 at full width: two equal largest logits (exactly 64)
    inside one tile, across tiles, across slices and, in steps of GROUP slices (which so few rows
    take only with a workspace for no more), across steps: the first wins."""
    _case("head ties")
    rng = np.random.default_rng(13)
    vocab, hidden = 151936, 256
    g = fused_head.GROUP * 8192
    pairs = [(4106, 4116), (1000, 5096), (100, 8242), (8191, 8192), (g - 1, g + 5),
             (vocab - 4000, vocab - 1)]
    w = (rng.standard_normal((vocab, hidden)) * 0.05).astype(np.float16)
    h = (rng.standard_normal((2 * len(pairs) + 4, hidden)) * 2).astype(np.float16)
    t = np.full(len(h), -100, np.int64)
    t[2 * len(pairs):] = rng.integers(0, vocab, 4)
    for i, (a, b) in enumerate(pairs):
        signs = rng.integers(0, 2, hidden) * 2 - 1
        w[a] = w[b] = (signs / 16).astype(np.float16)
        h[2 * i] = h[2 * i + 1] = (signs * 4).astype(np.float16)
        t[2 * i], t[2 * i + 1] = a, b
    res = _run(h, w, t, vchunk=8192)
    dev = [torch.from_numpy(x).to(DEV) for x in (h, w, t)]
    stepped = _head_ce_by_group(*dev, 8192, len(h), fused_head.GROUP)
    for r in (res, {k: v.cpu().numpy() for k, v in stepped.items()}):
        assert r["correct"][:2 * len(pairs)].tolist() == [True, False] * len(pairs)
        assert r["best_idx"][:2 * len(pairs)].tolist() == [a for a, _ in pairs for _ in range(2)]


def test_head_two_steps_of_more_than_eight_slices():
    """700 gradient rows at full width take steps of ten and nine slices: a second set of a step's
    statistics on top of stored ones, and an accumulator rescaled once. Every seventeenth row
    against the oracle, all of them against steps of GROUP slices."""
    _case("head steps of 10 and 9 slices")
    n, vocab, vchunk = 700, 151936, 8192
    h16, w16, t = exact_head_case(n, 64, vocab, 24)
    t = np.where(t >= 0, t, 7)
    dev = [torch.from_numpy(x).to(DEV) for x in (h16, w16, t)]
    out = fused_head.head_ce(*dev, vchunk, n)
    stepped = _head_ce_by_group(*dev, vchunk, n, fused_head.GROUP)
    for k in ("best_idx", "correct"):
        assert torch.equal(out[k], stepped[k])
    rows = np.arange(0, n, 17)
    ref = head_oracle.head_direct(h16[rows], w16, t[rows])
    scale = np.abs(ref["grad"]).max(1, keepdims=True)
    for res in (out, stepped):
        got = {k: v.cpu().numpy()[rows] for k, v in res.items()}
        assert np.all(np.abs(got["token_loss"] - ref["token_loss"]) <= 2e-5 + 2e-6 * ref["zmax"])
        assert np.all(np.abs(got["entropy"] - ref["entropy"]) <= 2e-5 + 1e-5 * ref["zmax"])
        assert np.array_equal(got["best_idx"], ref["best_idx"])
        assert np.all(np.abs(got["grad"] - ref["grad"]) <= 2e-3 * np.abs(ref["grad"]) + 2.0 ** -7 * scale)


@pytest.mark.parametrize("group", [None, 1])
def test_head_slices_wider_than_a_tile_per_lane(group):
    """Slices of more than 64 tiles (here 128, and a last one of 57): their statistics are taken in
    lane-strided loops, all slices in one step or one a step; rows past two 128-row blocks, some
    of them without a gradient."""
    _case(f"head wide slices, group {group}")
    n, n_grad, vocab, vchunk = 300, 270, 40000, 16384
    h16, w16, t = exact_head_case(n, 64, vocab, 25)
    t[n_grad:] = -100
    dev = [torch.from_numpy(x).to(DEV) for x in (h16, w16, t)]
    out = (fused_head.head_ce(*dev, vchunk, n_grad) if group is None
           else _head_ce_by_group(*dev, vchunk, n_grad, group))
    res = {k: v.float().cpu().numpy() if k == "grad" else v.cpu().numpy() for k, v in out.items()}
    n_lab = int((t >= 0).sum())
    res["loss"] = res["token_loss"].astype(np.float64).sum() / n_lab
    _check(res, h16, w16, t, vchunk, grad_scale=n_lab, what=f"group {group}")


@pytest.mark.parametrize("n", [1, 192, 193, 256, 257, 450])
def test_head_steps_of_many_slices(n):
    """Few rows take more than `group` slices per step (here all 22 of them, also more than the
    eight whose statistics are loaded at a time) and the last token tile of 256 rows may be partly
    empty, wavefront by wavefront (64 rows): losses, argmax and dH against the oracle, and the
    evaluation equal to the training pass bit for bit."""
    _case(f"head many slices n={n}")
    h16, w16, t = exact_head_case(n, 64, 2800, 30 + n)
    res = _run(h16, w16, t, vchunk=128)
    _check(res, h16, w16, t, 128, what=f"n={n}")
    dev = [torch.from_numpy(x).to(DEV) for x in (h16, w16, t)]
    out = fused_head.head_ce(*dev, vocab_chunk=128, need_grad=False)
    # the loss is 0 on unlabelled rows in both; rows are independent of their order
    np.testing.assert_array_equal(out["token_loss"].cpu().numpy(), res["token_loss"])
    np.testing.assert_array_equal(out["entropy"].cpu().numpy(), res["entropy"])
    np.testing.assert_array_equal(out["best_idx"].cpu().numpy(), res["best_idx"])


@pytest.mark.parametrize("vchunk", [1024, 16384])  # a tile per lane, and lane-strided loops
def test_head_tile_that_overflows_to_minus_infinity(vchunk):
    """Logits that all overflow fp16 to -inf in one statistics tile of 128 columns have probability
    0: losses, entropies and argmax are those of the vocabulary without them."""
    _case(f"head tile of -inf, vchunk={vchunk}")
    h16, w16, t = exact_head_case(40, 64, 9000, 21)
    h16[:, 0] = 256.0
    w16[:, 0] = 0.0
    gone = np.arange(9000) // 128 == 37
    w16[gone] = 0.0
    w16[gone, 0] = -512.0  # -131072
    t[gone[np.maximum(t, 0)] & (t >= 0)] = 5
    out = fused_head.head_ce(*(torch.from_numpy(x).to(DEV) for x in (h16, w16, t)),
                             vocab_chunk=vchunk, need_grad=False)
    kept = np.flatnonzero(~gone)
    place = np.cumsum(~gone) - 1
    ref = head_oracle.head_direct(h16, w16[kept], np.where(t >= 0, place[np.maximum(t, 0)], t))
    got = {k: v.cpu().numpy() for k, v in out.items() if v is not None}
    assert np.all(np.abs(got["token_loss"] - ref["token_loss"]) <= 2e-5 + 2e-6 * ref["zmax"])
    assert np.all(np.abs(got["entropy"] - ref["entropy"]) <= 2e-5 + 1e-5 * ref["zmax"])
    assert np.array_equal(got["best_idx"], kept[ref["best_idx"]])


@pytest.mark.parametrize("one_step", [True, False])
@pytest.mark.parametrize("where", ["first", "last"])
def test_head_gradient_of_confident_rows(where, one_step):
    """Rows that give their target, in the vocabulary's first or last slice, 18 more than the other
    logits' standard deviation of 1.5, with weight rows around a common mean: dH is the sum of
    151935 small weights times their rows. Every logit is exact in fp16 (multiples of 1/64 below 32).
    The bound, per element: fp16's rounding of dH, of P, of the tile's factor and of their product
    (2^-11 each, of the sum of p |w|); P's subnormals in the target's own tile (2^-25 each); the fp32
    sums, whose rounding errors (2^-24 of a partial sum of at most |w[target]|, one per MFMA step
    and part) add up at random."""
    _case(f"head confident rows, target in the {where} slice, one step: {one_step}")
    rng = np.random.default_rng(14)
    vocab, hidden, n, vchunk = 151936, 64, 6, 8192
    h = np.stack([rng.permutation(np.repeat([1.0, -1.0], hidden // 2)) for _ in range(n)])
    w = 0.25 + np.rint(rng.standard_normal((vocab, hidden)) * 12) / 64
    t = np.arange(n) * 37 + (100 if where == "first" else vocab - 1000)
    w[t] += h * (18 / 64)
    h, w = h.astype(np.float16), w.astype(np.float16)
    ref = head_oracle.head_direct(h, w, t)
    z = head_oracle.logits16(h, w).astype(np.float64)
    assert np.array_equal(z, h.astype(np.float64) @ w.astype(np.float64).T)
    dev = [torch.from_numpy(x).to(DEV) for x in (h, w, t)]
    if one_step:
        got = fused_head.head_ce(*dev, vocab_chunk=vchunk, n_grad=n)["grad"]
    else:
        got = _head_ce_by_group(*dev, vchunk, n, fused_head.GROUP)["grad"]
    p = np.exp(z - z.max(1)[:, None])
    p /= p.sum(1)[:, None]
    p[np.arange(n), t] = 0
    absw = np.abs(w.astype(np.float64))
    steps = vocab / 16 + 48
    bound = (2.0 ** -11 * np.abs(ref["grad"]) + 2.0 ** -25 + 3 * 2.0 ** -11 * (p @ absw)
             + 127 * 2.0 ** -25 * absw.max() + 4 * np.sqrt(steps) * 2.0 ** -24 * absw[t])
    err = np.abs(got.double().cpu().numpy() - ref["grad"])
    rel = np.linalg.norm(err, axis=1) / np.linalg.norm(ref["grad"], axis=1)
    print(f"[head] p {1 - p.sum(1).max():.4f}, relative error of dH {rel.max():.2e}, "
          f"of the bound {(err / bound).max():.2f}", flush=True)
    assert np.all(err <= bound)


@pytest.mark.parametrize("n_grad", [0, 70])
def test_head_workspace_of_the_smaller_step(n_grad):
    """A workspace that holds `group` slices a step but not more (one kept from another call) still
    serves: the loop takes `group` at a time, with the same losses and dH to the rescales'
    rounding (each step's factors are rounded to fp16)."""
    group, vchunk, vocab = 3, 128, 9 * 128
    h16, w16, t = exact_head_case(70, 64, vocab, 50)
    h, w, tt = [torch.from_numpy(x).to(DEV) for x in (h16, w16, t)]
    full = fused_head.head_ce(h, w, tt, vchunk, n_grad, n_grad > 0, group)
    got = _head_ce_by_group(h, w, tt, vchunk, n_grad, group)
    assert torch.equal(got["best_idx"], full["best_idx"])
    assert torch.equal(got["token_loss"], full["token_loss"])
    if n_grad:  # one fp16 rounding of each column's factor, one of dH
        ref = full["grad"].double()
        bound = 2.0 ** -10 * (ref.abs() + w.double().abs().max())
        assert bool(((got["grad"].double() - ref).abs() <= bound).all())


def test_head_config4_full_size_every_row():
    """Config 4: H [2048, 1536] ~N(0, 1), W [151936, 1536] ~N(0, 0.02), 10% ignored, 8192-column
    slices. Every row is checked against the float64 closed form (each row's outputs depend on
    that row only, so the oracle runs over chunks of 256 rows), correctness exact except near
    ties."""
    _case("head config4, every row")
    d = workloads.head_inputs()
    h16, w16, t = d["hidden"].numpy(), d["weight"].numpy(), d["targets"].numpy()
    res = _run(h16, w16, t, vchunk=8192, grad_scale=1.0)
    n_lab = int((t >= 0).sum())
    w64 = w16.astype(np.float64)
    sum_ours = sum_ref = 0.0
    fragile_rows = 0
    for r0 in range(0, len(t), 256):
        rows = slice(r0, min(r0 + 256, len(t)))
        ref = head_oracle.head_direct(h16[rows], w64, t[rows])
        zmax = ref["zmax"]
        ulp = 2.0 ** (np.floor(np.log2(zmax)) - 10)
        sub = {k: res[k][rows] for k in ("token_loss", "entropy", "correct", "best_idx", "grad")}
        # the reference's random-style bounds (solution/test_fuzz.py:293-297)
        assert np.all(np.abs(sub["token_loss"] - ref["token_loss"]) <= 2e-5 + 2e-6 * zmax + 8 * ulp), r0
        assert np.all(np.abs(sub["entropy"] - ref["entropy"]) <= 2e-5 + 1e-5 * zmax + 16 * ulp), r0
        lab = t[rows] >= 0
        sum_ours += float(sub["token_loss"][lab].astype(np.float64).sum())
        sum_ref += float(ref["token_loss"][lab].sum())
        # near ties: the top-2 fp16 logits within 2 ulps may flip with the summation order
        z = head_oracle.logits16(h16[rows], w16).astype(np.float32)
        top2 = np.sort(z, 1)[:, -2:]
        fragile = (top2[:, 1] - top2[:, 0]) <= 2 * 2.0 ** (np.floor(np.log2(np.abs(top2[:, 1]))) - 10)
        fragile_rows += int(fragile.sum())
        assert np.all((sub["best_idx"] == ref["best_idx"]) | fragile), r0
        assert np.all((sub["correct"] == ref["correct"]) | fragile), r0
        g_ref = ref["grad"] / n_lab
        scale = np.abs(g_ref).max()
        assert np.all(np.abs(sub["grad"] - g_ref) <= 2e-3 * np.abs(g_ref) + 2.0 ** -7 * scale), r0
    print(f"[head config4] {len(t)} rows, {n_lab} labelled, {fragile_rows} near ties", flush=True)
    assert abs(sum_ours - sum_ref) <= 1e-4 * abs(sum_ref)  # CE within 1e-4 relative
    total = res["token_loss"].astype(np.float64).sum() / n_lab
    assert abs(res["loss"] - total) <= 1e-5 * total
    assert abs(res["loss"] - sum_ref / n_lab) <= 1e-4 * sum_ref / n_lab


def test_head_weight_transpose_and_cache():
    """talm_head_weight_t: exact transpose with zero columns past the vocabulary. head_weights:
    the fp16 copy of an fp32 output weight is made once per weight version and rebuilt after an
    in-place update; an fp16 weight is used as it lies."""
    _case("head weight_t + cache")
    w = torch.randn(1003, 136, device=DEV).half()
    wt = torch.empty(136, 1024, dtype=torch.float16, device=DEV)
    torch.ops.talm.head_weight_t(w, wt)
    assert torch.equal(wt[:, :1003], w.t())
    assert bool(torch.all(wt[:, 1003:] == 0))
    assert fused_head.head_weights(w).data_ptr() == w.data_ptr()
    w32 = torch.randn(1003, 136, device=DEV)
    a = fused_head.head_weights(w32)
    assert fused_head.head_weights(w32) is a and torch.equal(a, w32.half())
    w32.mul_(2)
    c = fused_head.head_weights(w32)
    assert c is not a and torch.equal(c, w32.half())