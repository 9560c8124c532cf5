"""The five BASELINE workloads at their full sizes on the GPU.

The oracle cannot finish these sizes in seconds, so parity is checked (a) against the oracle on a
random subsample of queries and of touched entities, and (b) through size-independent properties:
bit-exact integer invariants of the segment plan, untouched rows staying bit-identical (row
checksums), exact linearity of the backward in the upstream gradient (scaling by 2 is exact in
fp32), and run-to-run determinism."""
import gc

import numpy as np
import pytest
import torch

import bench
from oracle import oracle as orc
from tests.util import REL_F32, assert_close

pytestmark = pytest.mark.gpu


def _oracle_rows(table, ids):
    return table[torch.as_tensor(ids, device=table.device)].cpu().numpy().astype(np.float64)


def _oracle_segment_gradient(model, row, q1, q2, pairs, k, gs, cen, chunk=16384):
    """Float64 oracle gradient of one entity row summed over all pairs of its segment, and the sum of the
    terms' magnitudes.  The segment is fed to the oracle in chunks (the hottest cfg5 ids own up to ~470,000
    pairs: one oracle call over all of them would need gigabytes of repeated rows), partial sums added in
    float64 in pair order."""
    row = row.cpu().numpy().astype(np.float64)
    want = np.zeros(row.shape[-1])
    sum_abs = np.zeros(row.shape[-1])
    flat_gs = gs.reshape(-1)
    for lo in range(0, pairs.numel(), chunk):
        part = pairs[lo: lo + chunk]
        pb = part // k
        e = np.broadcast_to(row, (part.numel(), 1, row.shape[-1]))
        a1 = q1[pb].cpu().numpy().astype(np.float64)[:, None]
        a2 = None if q2 is None else q2[pb].cpu().numpy().astype(np.float64)[:, None]
        og = flat_gs[part].cpu().numpy().astype(np.float64)[:, None]
        g_rows, _, _ = orc.score_backward(model, og, np.ascontiguousarray(e), a1, a2, cen)
        want += g_rows.sum(axis=(0, 1))
        sum_abs += np.abs(g_rows).sum(axis=(0, 1))
    return want, sum_abs


@pytest.mark.parametrize("cfg_id", [1, 2, 3, 4, 5])
def test_full_size_workload(cfg_id):
    from smore_amd import fused
    cfg = bench.CONFIGS[cfg_id]
    dev = torch.device("cuda:0")
    gc.collect()
    torch.cuda.empty_cache()    # what an earlier test of this size has released is still held by the caching allocator
    free, _ = torch.cuda.mem_get_info()
    need = cfg["n"] * bench.row_len(cfg) * 4 * (3 if cfg["adam"] else 1) + (4 << 30)
    if free < need:
        pytest.skip(f"needs {need >> 30} GiB of HBM, {free >> 30} free")
    table, q1, q2, idx, gs = bench.make_inputs(cfg, dev, 20240 + cfg_id)
    model, n, b, k = cfg["model"], cfg["n"], cfg["b"], cfg["k"]
    params = fused.score_params(cfg["gamma"], cfg["cen"])
    err = fused.new_error_flag(dev)
    rng = np.random.default_rng(cfg_id)

    # ---- plan: integer invariants, bit-exact
    plan = fused.build_plan(idx, n, want_inverse=True, err_flag=err)
    u = plan.n_uniq
    uniq_t = torch.unique(idx)
    assert u == uniq_t.numel() and torch.equal(plan.uniq, uniq_t)
    seg = plan.seg_start[: u + 1].long()
    assert seg[0].item() == 0 and seg[-1].item() == b * k and bool((seg[1:] > seg[:-1]).all())
    flat = idx.reshape(-1)
    assert torch.equal(flat[plan.order.long()], plan.sorted_ids.long())
    assert torch.equal(plan.uniq[plan.inverse], flat)
    order = plan.order.long()
    same_seg = plan.sorted_ids[1:] == plan.sorted_ids[:-1]
    assert bool((order[1:][same_seg] > order[:-1][same_seg]).all()), "pairs inside a segment must stay in pair order"

    # ---- forward + query backward: oracle on a sample of queries
    score = fused.score_forward(model, table, idx, q1, q2, params, err)
    gq1, gq2 = fused.score_backward_query(model, table, idx, q1, q2, score, gs, params)
    assert err.item() == 0
    qs = np.sort(rng.choice(b, size=min(b, 24), replace=False))
    ids_s = idx[qs].cpu().numpy()
    rows = _oracle_rows(table, ids_s.reshape(-1)).reshape(len(qs), k, -1)
    oq1 = q1[qs].cpu().numpy().astype(np.float64)[:, None]
    oq2 = None if q2 is None else q2[qs].cpu().numpy().astype(np.float64)[:, None]
    ogs = gs[qs].cpu().numpy().astype(np.float64)
    assert_close(score[qs].cpu().numpy(), orc.score_forward(model, rows, oq1, oq2, cfg["gamma"], cfg["cen"]),
                 REL_F32, "score sample", rms_floor=False)
    _, o1, o2 = orc.score_backward(model, ogs, rows, oq1, oq2, cfg["cen"])
    assert_close(gq1[qs].cpu().numpy(), o1[:, 0], REL_F32, "gq1 sample")
    if q2 is not None:
        assert_close(gq2[qs].cpu().numpy(), o2[:, 0], REL_F32, "gq2 sample")

    # ---- linearity and determinism of the query backward (exact)
    g2a, g2b = fused.score_backward_query(model, table, idx, q1, q2, score, gs * 2, params)
    assert torch.equal(g2a, gq1 * 2) and (q2 is None or torch.equal(g2b, gq2 * 2))

    # ---- entity backward: merged gradient for a sample of entities against brute force
    sample_u = np.unique(np.concatenate([rng.choice(u, size=min(u, 48), replace=False), np.arange(min(u, 3))]))
    merged = torch.empty((u, table.shape[1]), device=dev) if not cfg["adam"] else None
    row_sum_before = table.sum(dim=1) if cfg["adam"] else None
    w_before = {int(plan.uniq[j]): table[int(plan.uniq[j])].clone() for j in sample_u}
    if cfg["adam"]:
        m = torch.zeros_like(table)
        v = torch.zeros_like(table)
        fused.score_backward_entity(model, plan, table, q1, q2, score, gs, params, m=m, v=v,
                                    adam=fused.adam_params(cfg["lr"], 1))
    else:
        fused.score_backward_entity(model, plan, table, q1, q2, score, gs, params, merged=merged)
        merged_again = torch.empty_like(merged)
        fused.score_backward_entity(model, plan, table, q1, q2, score, gs, params, merged=merged_again)
        assert torch.equal(merged, merged_again), "entity pass must be deterministic"
    seg_np = seg.cpu().numpy()
    hottest = 0
    for j in sample_u:
        pairs = plan.order[seg_np[j]: seg_np[j + 1]].long()
        eid = int(plan.uniq[j])
        hottest = max(hottest, pairs.numel())
        want, sum_abs = _oracle_segment_gradient(model, w_before[eid], q1, q2, pairs, k, gs, cfg["cen"])
        e = w_before[eid].cpu().numpy().astype(np.float64)[None, None, :]
        if cfg["adam"]:
            got_m = m[eid].cpu().numpy().astype(np.float64)
            assert_close(got_m, 0.1 * want, REL_F32, f"first moment of entity {eid}", sum_abs=0.1 * sum_abs)
            wn, mn, vn = e[0, 0][None].copy(), np.zeros((1, e.shape[-1])), np.zeros((1, e.shape[-1]))
            orc.adam_rows(wn, mn, vn, np.array([0]), (got_m / 0.1)[None], cfg["lr"], 1)
            assert_close(table[eid].cpu().numpy(), wn[0], REL_F32, f"weights of entity {eid}")
        else:
            assert_close(merged[j].cpu().numpy(), want, REL_F32, f"merged gradient of entity {eid}", sum_abs=sum_abs)

    if cfg_id == 5:   # Zipf ids: the sample must have covered the long-segment kernels (tiles + fix-up)
        assert hottest > 100000, hottest

    # ---- touched-row set: only rows of uniq may change (row checksums, exact)
    if cfg["adam"]:
        changed = (table.sum(dim=1) != row_sum_before).nonzero().flatten()
        assert bool(torch.isin(changed, plan.uniq).all()), "a row outside the touched set changed"
        touched_m = (m.abs().sum(dim=1) != 0).nonzero().flatten()
        assert bool(torch.isin(touched_m, plan.uniq).all())
        # every touched row gets a non-zero moment unless its upstream gradients are exactly 0.0
        # (torch.randn does return a few exact zeros among 4M samples)
        assert u - touched_m.numel() <= int((gs == 0).sum().item())
        assert changed.numel() > 0.9 * u  # a row sum can stay put when its +-lr moves cancel

    # ---- the path bench.py times, as a second step on the state the first one left: forward that saves the
    # sign codes (box) + one-call backward (query gradients, entity pass, optimizer), against the separate
    # calls (query gradients) and the oracle (sampled entities)
    if not cfg["adam"]:
        # whichever kernel finishes a segment: bit-identical rows for the sign-coded models, and for the
        # others the same sum up to the rounding of differently contracted multiply-adds
        codes = fused.new_codes(model, table, idx, q1)
        score2 = fused.score_forward(model, table, idx, q1, q2, params, err, codes=codes)
        assert torch.equal(score2, score)
        merged_one_call = torch.empty_like(merged)
        f1, f2 = fused.score_backward_fused(model, plan, table, idx, q1, q2, score2, gs, params,
                                            merged=merged_one_call, codes=codes)
        if codes is not None:
            assert torch.equal(merged_one_call, merged), "one-call merged gradient differs from the entity pass"
        else:
            assert_close(merged_one_call.cpu().numpy(), merged.cpu().numpy(), 1e-6, "one-call merged gradient")
        assert_close(f1.cpu().numpy(), gq1.cpu().numpy(), 1e-6, "one-call gq1")
        if q2 is not None:
            assert_close(f2.cpu().numpy(), gq2.cpu().numpy(), 1e-6, "one-call gq2")
    if cfg["adam"]:
        codes = fused.new_codes(model, table, idx, q1)
        score2 = fused.score_forward(model, table, idx, q1, q2, params, err, codes=codes)
        assert torch.equal(score2, fused.score_forward(model, table, idx, q1, q2, params, err))
        r1, r2 = fused.score_backward_query(model, table, idx, q1, q2, score2, gs, params)
        eids = [int(plan.uniq[j]) for j in sample_u]
        before = {e_: (table[e_].clone(), m[e_].clone(), v[e_].clone()) for e_ in eids}
        f1, f2 = fused.score_backward_fused(model, plan, table, idx, q1, q2, score2, gs, params, m=m, v=v,
                                            adam=fused.adam_params(cfg["lr"], 2), codes=codes)
        assert_close(f1.cpu().numpy(), r1.cpu().numpy(), 1e-6, "one-call gq1")
        if q2 is not None:
            assert_close(f2.cpu().numpy(), r2.cpu().numpy(), 1e-6, "one-call gq2")
        for j, eid in zip(sample_u, eids):
            pairs = plan.order[seg_np[j]: seg_np[j + 1]].long()
            w1, m1, v1 = (x.cpu().numpy().astype(np.float64) for x in before[eid])
            want, sum_abs = _oracle_segment_gradient(model, before[eid][0], q1, q2, pairs, k, gs, cfg["cen"])
            got_m = m[eid].cpu().numpy().astype(np.float64)
            assert_close(got_m, 0.9 * m1 + 0.1 * want, REL_F32, f"step 2 first moment of entity {eid}",
                         sum_abs=0.1 * sum_abs + 0.9 * np.abs(m1))
            wn, mn, vn = w1[None].copy(), m1[None].copy(), v1[None].copy()
            orc.adam_rows(wn, mn, vn, np.array([0]), ((got_m - 0.9 * m1) / 0.1)[None], cfg["lr"], 2)
            assert_close(table[eid].cpu().numpy(), wn[0], REL_F32, f"step 2 weights of entity {eid}")
            assert_close(v[eid].cpu().numpy(), vn[0], REL_F32, f"step 2 second moment of entity {eid}",
                         sum_abs=np.full_like(w1, 1e-12), rms_floor=False)


@pytest.mark.parametrize("n_pairs", [4096 * 1025, 4096 * 1025 + 4096, 18 * 1024 * 256 + 5, 6_000_000])
def test_plan_at_pair_counts_beyond_256_tiles_of_16_rounds(n_pairs):
    """A step that scores positives beside the negatives holds B x (1 + K) pairs (kg_reasoning.py:340-355), with
    anchors B more: just past the 4,194,304 the radix passes cover with 16 elements per thread and one tile per CU.
    They then take 17 or 18 per thread; beyond that, more tiles.  Integer invariants against torch, bit-exact."""
    from smore_amd import fused
    n = 86_054_151
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n_pairs % 1000)
    ids = bench.zipf_ids(n, (n_pairs,), 1.1, gen, torch.device("cuda"))
    plan = fused.build_plan(ids, n, want_inverse=True)
    uniq_t, inverse_t = torch.unique(ids, return_inverse=True)
    assert plan.n_uniq == uniq_t.numel() and torch.equal(plan.uniq, uniq_t)
    assert torch.equal(plan.inverse, inverse_t)
    assert torch.equal(ids[plan.order.long()], plan.sorted_ids.long())
    assert bool((plan.sorted_ids[1:] >= plan.sorted_ids[:-1]).all())
    order = plan.order.long()
    same_seg = plan.sorted_ids[1:] == plan.sorted_ids[:-1]
    assert bool((order[1:][same_seg] > order[:-1][same_seg]).all()), "pairs inside a segment must stay in pair order"
    counts = torch.bincount(inverse_t, minlength=uniq_t.numel())
    seg = plan.seg_start[: plan.n_uniq + 1].long()
    assert torch.equal(seg[1:] - seg[:-1], counts)
    alone = plan.pair_seg < 0
    assert int(alone.sum().item()) == int((counts == 1).sum().item())


def test_plan_around_the_tile_geometry_boundaries():
    """Pair counts on both sides of every change of the radix passes' geometry near one tile per CU (16, 17, 18
    elements per thread, then a second round of tiles), uniform 27-bit ids: sorted order, stability and segment
    table against torch's stable sort."""
    from smore_amd import fused
    n = 86_054_151
    gen = torch.Generator(device="cuda")
    gen.manual_seed(99)
    per = 1024 * 256
    # (and of the emit kernel's: one sorted position per thread up to 2^18 positions, four up to 2^20, sixteen beyond)
    for n_pairs in (4097, per - 1, per, per + 1, 4 * per - 1, 4 * per, 4 * per + 1,
                    16 * per - 1, 16 * per, 16 * per + 1, 17 * per, 17 * per + 1, 18 * per - 1, 18 * per, 18 * per + 1,
                    18 * per + 18 * 1024, 19 * per + 7):
        ids = torch.randint(0, n, (n_pairs,), device="cuda", generator=gen)
        ids[: n_pairs // 50] = ids[0]                                  # one long segment as well
        plan = fused.build_plan(ids, n)
        want_ids, want_order = torch.sort(ids, stable=True)
        assert torch.equal(plan.sorted_ids.long(), want_ids), n_pairs
        assert torch.equal(plan.order.long(), want_order), n_pairs
        heads = torch.ones(n_pairs, dtype=torch.bool, device="cuda")
        heads[1:] = want_ids[1:] != want_ids[:-1]
        assert plan.n_uniq == int(heads.sum().item())
        assert torch.equal(plan.seg_start[: plan.n_uniq].long(), torch.nonzero(heads).reshape(-1))


@pytest.mark.parametrize("rounds", [2, 8])
@pytest.mark.parametrize("n", [40_000, 900_000])
def test_plan_between_the_forms_of_the_radix_pass(rounds, n):
    """Pair counts around the lengths of a thread's stretch at which another form of the pass takes over, two-pass
    plans (16- and 20-bit ids): sorted order, stability and segment table against torch's stable sort."""
    from smore_amd import fused
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rounds)
    per = 1024 * 256
    for n_pairs in (rounds * per - 1, rounds * per, rounds * per + 1):
        ids = torch.randint(0, n, (n_pairs,), device="cuda", generator=gen)
        ids[: n_pairs // 50] = ids[0]
        plan = fused.build_plan(ids, n)
        want_ids, want_order = torch.sort(ids, stable=True)
        assert torch.equal(plan.sorted_ids.long(), want_ids) and torch.equal(plan.order.long(), want_order), n_pairs
        heads = torch.ones(n_pairs, dtype=torch.bool, device="cuda")
        heads[1:] = want_ids[1:] != want_ids[:-1]
        assert plan.n_uniq == int(heads.sum().item())
        assert torch.equal(plan.seg_start[: plan.n_uniq].long(), torch.nonzero(heads).reshape(-1))


def test_plan_beyond_4096_tiles():
    """More than 4096 tiles of 18 elements per thread: the look-back's three levels end and the chain of prefixes
    over stretches of 4096 tiles takes over.  Sorted order, stability and segment table against torch's stable sort."""
    from smore_amd import fused
    n = 86_054_151
    n_pairs = 4096 * 18 * 1024 + 3 * 18 * 1024 + 77
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4097)
    ids = torch.randint(0, n, (n_pairs,), device="cuda", generator=gen)
    ids[: n_pairs // 64] = ids[0]
    plan = fused.build_plan(ids, n)
    want_ids, want_order = torch.sort(ids, stable=True)
    assert torch.equal(plan.sorted_ids.long(), want_ids)
    assert torch.equal(plan.order.long(), want_order)
    heads = torch.ones(n_pairs, dtype=torch.bool, device="cuda")
    heads[1:] = want_ids[1:] != want_ids[:-1]
    assert plan.n_uniq == int(heads.sum().item())
    assert torch.equal(plan.seg_start[: plan.n_uniq].long(), torch.nonzero(heads).reshape(-1))


def test_full_size_dropin_flow():
    """The 86M-entity step as SMORE's own code reaches it: lookup handles for positives and negatives, the box
    model's cal_logit (box.py:157-164) on them, backward, apply_grad -- nothing but the reference's call sequence
    (kg_reasoning.py:298-307, 340-355; train_process.py:172-220).  No lookup may be materialised and no logit may
    leave the fused scorer; logits, relation gradients and the Adam state of sampled entities (the three hottest
    included) against the float64 oracle; rows outside the touched set bit-identical."""
    import types
    from smore_amd.embedding.embed_optimizer import AdamEmbedOptimizer
    from smore_amd.embedding.sparse_embed import SparseEmbedding
    from smore_amd.torchext.ext_ops import box_dist_in, box_dist_out
    cfg = bench.CONFIGS[5]
    dev = torch.device("cuda:0")
    gc.collect()
    torch.cuda.empty_cache()    # what an earlier test of this size has released is still held by the caching allocator
    free, _ = torch.cuda.mem_get_info()
    need = cfg["n"] * bench.row_len(cfg) * 4 * 3 + (6 << 30)
    if free < need:
        pytest.skip(f"needs {need >> 30} GiB of HBM, {free >> 30} free")
    table, q1, q2, idx, gs = bench.make_inputs(cfg, dev, 20245)
    n, b, k, lr = cfg["n"], cfg["b"], cfg["k"], cfg["lr"]
    rng = np.random.default_rng(55)
    emb = SparseEmbedding(8, cfg["dim"])
    emb.embedding = torch.nn.Parameter(table, requires_grad=True)
    emb.num_rows = n
    opt = AdamEmbedOptimizer(types.SimpleNamespace(optim_mode="(aggr,adam,gpu,False,5)", share_optim_stats=True), emb, 0)
    gamma = torch.nn.Parameter(torch.tensor([cfg["gamma"]], device=dev), requires_grad=False)
    rel_c, rel_o = q1.clone().requires_grad_(True), q2.clone().requires_grad_(True)
    pos = idx[:, 7].contiguous()
    gp = gs[:, :1].contiguous()

    def cal_logit(rows, center, offset):
        return torch.max(gamma - box_dist_out(rows, center, offset) - cfg["cen"] * box_dist_in(rows, center, offset), dim=1)[0]

    ids_all = torch.cat([pos[:, None], idx], dim=1)
    gs_all = torch.cat([gp, gs], dim=1)
    uniq = torch.unique(ids_all)
    sample = np.unique(np.concatenate([rng.choice(uniq.numel(), size=40, replace=False), np.arange(3)]))
    sample_ids = uniq[torch.as_tensor(sample, device=dev)].tolist()
    w_before = {e: table[e].clone() for e in sample_ids}
    row_sum_before = table.detach().sum(dim=1)
    qs = np.sort(rng.choice(b, size=16, replace=False))           # queries whose logits and gradients the oracle checks
    qs_t = torch.as_tensor(qs, device=dev)
    rows_q = table.detach()[ids_all[qs_t]].cpu().numpy().astype(np.float64)      # [16, 1 + K, row], before the update

    opt.zero_grad()
    center, offset = rel_c.view(b, 1, 1, -1), rel_o.view(b, 1, 1, -1)
    p_rows = emb(pos, "positive_entity")
    n_rows = emb(idx.view(-1), "negative_entity")
    lp = cal_logit(p_rows.unsqueeze(1), center, offset)
    ln = cal_logit(n_rows.view(b, k, -1), center, offset)
    ((lp * gp).sum() + (ln * gs).sum()).backward()
    assert opt.stats == dict(fused_launches=1, materialized_lookups=0, dense_fallbacks=0, per_record_merges=0)
    opt.apply_grad(lr)
    opt.check_ids()
    assert opt.stats["per_record_merges"] == 0 and opt.stats["materialized_lookups"] == 0

    got_logit = torch.cat([lp, ln], dim=1).detach()

    # entity side: first moment and weights of the sampled entities from their saved rows, all their pairs
    flat_ids = ids_all.reshape(-1)
    m = emb.state_sum_fo
    hottest = 0
    for e in sample_ids:
        pairs = (flat_ids == e).nonzero().flatten()
        hottest = max(hottest, pairs.numel())
        want, sum_abs = _oracle_segment_gradient("box", w_before[e], q1, q2, pairs, k + 1, gs_all, cfg["cen"])
        got_m = m[e].cpu().numpy().astype(np.float64)
        assert_close(got_m, 0.1 * want, REL_F32, f"drop-in flow: first moment of entity {e}", sum_abs=0.1 * sum_abs)
        w0 = w_before[e].cpu().numpy().astype(np.float64)
        wn, mn, vn = w0[None].copy(), np.zeros((1, w0.size)), np.zeros((1, w0.size))
        orc.adam_rows(wn, mn, vn, np.array([0]), (got_m / 0.1)[None], lr, 1)
        assert_close(table[e].detach().cpu().numpy(), wn[0], REL_F32, f"drop-in flow: weights of entity {e}")
        # this entity's logits, from its saved row, for up to 64 of its pairs
        part = pairs[:64]
        pb = (part // (k + 1)).cpu().numpy()
        erow = np.broadcast_to(w0, (part.numel(), 1, w0.size))
        a1 = q1[torch.as_tensor(pb, device=dev)].cpu().numpy().astype(np.float64)[:, None]
        a2 = q2[torch.as_tensor(pb, device=dev)].cpu().numpy().astype(np.float64)[:, None]
        want_logit = orc.score_forward("box", np.ascontiguousarray(erow), a1, a2, cfg["gamma"], cfg["cen"])[:, 0]
        assert_close(got_logit.reshape(-1)[part].cpu().numpy(), want_logit, REL_F32, f"drop-in flow: logits of entity {e}",
                     rms_floor=False)
    assert hottest > 100000, hottest

    # logits and relation gradients of the sampled queries
    oq1 = q1[qs_t].cpu().numpy().astype(np.float64)[:, None]
    oq2 = q2[qs_t].cpu().numpy().astype(np.float64)[:, None]
    assert_close(got_logit[qs_t].cpu().numpy(), orc.score_forward("box", rows_q, oq1, oq2, cfg["gamma"], cfg["cen"]),
                 REL_F32, "drop-in flow: logits of sampled queries", rms_floor=False)
    _, o1, o2 = orc.score_backward("box", gs_all[qs_t].cpu().numpy().astype(np.float64), rows_q, oq1, oq2, cfg["cen"])
    assert_close(rel_c.grad[qs_t].cpu().numpy(), o1[:, 0], REL_F32, "drop-in flow: center gradient of sampled queries")
    assert_close(rel_o.grad[qs_t].cpu().numpy(), o2[:, 0], REL_F32, "drop-in flow: offset gradient of sampled queries")

    # touched-row set: only rows of the step's ids may have changed
    changed = (table.detach().sum(dim=1) != row_sum_before).nonzero().flatten()
    assert bool(torch.isin(changed, uniq).all()), "a row outside the touched set changed"
