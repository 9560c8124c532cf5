"""Filtered ranks of the answers of a batch of queries among ALL entities, as test_step_mp computes
them (smore/training/train_process.py:112-160), on the streaming HIP scan instead of
`argsort` over the [1, nentity] logit row."""
import ctypes
from itertools import chain

import numpy as np
import torch

from .. import _lib
from ..fused import MODELS, _dims, _on, _ptr, _stream, _workspace


def _plain(values):
    """Integers of a list, tuple, range, array or host tensor as a one-dimensional int64 array, None for anything else."""
    try:
        a = np.asarray(values)
    except (TypeError, ValueError, RuntimeError):       # device tensors, sequences of them, ragged lists
        return None
    return a.astype(np.int64) if a.ndim == 1 and (a.dtype.kind == "i" or not a.size) else None


def _int64(ids):
    """Entity ids of one answer list as an int64 array: what torch takes for integers and nothing else (no strings, no dates)."""
    a = _plain(ids)
    return torch.as_tensor(list(ids), dtype=torch.int64).cpu().numpy() if a is None else a


def _counts(n_hard):
    """Hard-answer counts as an int32 tensor, likewise."""
    a = _plain(n_hard) if isinstance(n_hard, (list, tuple)) else None
    if a is None or (a.size and (a.min() < 0 or a.max() > 0x7fffffff)):
        return torch.as_tensor(n_hard, dtype=torch.int32).reshape(-1)
    return torch.from_numpy(a.astype(np.int32))


def _staging(count, dtype, dev):
    """Host memory, and whether a copy from it to the device need not be waited for (pinned: it is given out again once that
    copy has passed).  Under graph capture pageable memory: such a call is refused, a replay would copy whatever then lies
    there."""
    pinned = dev.type == "cuda" and not torch.cuda.is_current_stream_capturing()
    return torch.empty(count, dtype=dtype, pin_memory=pinned), pinned


def _counts_on(counts, dev):
    if counts.device.type != "cpu":
        return counts.to(dev)
    host, pinned = _staging(counts.numel(), torch.int32, dev)
    host.copy_(counts)
    return host.to(dev, non_blocking=pinned)


def _one_array(lists):
    """The ids of all answer lists in a row, where they are plain lists of integers; None otherwise."""
    if not all(type(ids) in (list, tuple) for ids in lists):
        return None
    return _plain(list(chain.from_iterable(lists)))


def filtered_ranks(model, table, q1, q2, params, easy_answers, hard_answers, branches=1):
    """model: score model name; table [N,row]; q1/q2 [B,dim] (q2 None for l1/l2); params from
    fused.score_params (gamma, cen, regularizer); easy_answers / hard_answers: per query a sequence of
    entity ids (disjoint, train_process.py:139).  Returns per query a pair of int64 tensors (device):
    the filtered ranks (1-based) of its hard answers, in the order given, and of its easy answers.
    branches > 1: union queries, q1/q2 [B, branches, dim]; an entity's logit is the maximum over the branches
    (custom_cal_logit, box.py:163)."""
    if q1.numel() % (branches * q1.shape[-1]):
        raise _lib.SmxError("q1 must hold `branches` rows per query")
    b = q1.numel() // (branches * q1.shape[-1])
    if len(easy_answers) != b or len(hard_answers) != b:
        raise _lib.SmxError("one answer list per query is needed")
    n = table.shape[0]
    sizes = [(len(e), len(h)) for e, h in zip(easy_answers, hard_answers)]
    a = max(1, max(ne + nh for ne, nh in sizes))
    # ids [B, A] and the counts behind them travel to the device as one array, which nothing waits for
    host, pinned = _staging(b * a + (b + 1) // 2, torch.int64, table.device)
    packed = host.numpy()
    packed[:] = 0
    ids, counts = packed[: b * a].reshape(b, a), packed[b * a:].view(np.int32)
    counts[:b] = [ne + nh for ne, nh in sizes]
    flat = _one_array([x for pair in zip(easy_answers, hard_answers) for x in pair])
    if flat is not None:
        ids[np.arange(a) < counts[:b, None]] = flat
    else:
        for i, (e, h) in enumerate(zip(easy_answers, hard_answers)):
            ne, nh = sizes[i]
            if ne:
                ids[i, :ne] = _int64(e)
            if nh:
                ids[i, ne: ne + nh] = _int64(h)
    used = np.arange(a) < counts[:b, None]
    if ids.min() < 0 or ids.max() >= n:
        raise IndexError("answer id outside the entity table")
    ordered = np.sort(np.where(used, ids, -1 - np.arange(a)), axis=1)      # (unused slots: distinct values of their own)
    if (ordered[:, 1:] == ordered[:, :-1]).any():
        raise _lib.SmxError("an entity is listed twice among the answers of one query")
    dev = table.device
    packed = host.to(dev, non_blocking=pinned)
    ids, counts = packed[: b * a].view(b, a), packed[b * a:]
    q1c = q1.reshape(b * branches, -1).contiguous()
    q2c = None if q2 is None else q2.reshape(b * branches, -1).contiguous()
    _, _, dim = _dims(model, table, ids, q1c[:b], None if q2c is None else q2c[:b])
    ranks = torch.empty((b, a), dtype=torch.int64, device=dev)
    with _on(dev):
        ws = _workspace(_lib.load().smx_filtered_ranks_workspace_bytes(MODELS[model], b, branches, a, dim), dev)
        _lib.call("smx_filtered_ranks", MODELS[model], _stream(table), _ptr(table), n, _ptr(q1c), _ptr(q2c), b, branches,
                  dim, ctypes.byref(params), _ptr(ids), _ptr(counts), a, None, _ptr(ranks), _ptr(ws), ws.numel())
    pieces = torch.split(ranks.view(-1), [s for ne, nh in sizes for s in (ne, nh, a - ne - nh)])   # easy, hard, unused
    return [(pieces[3 * i + 1], pieces[3 * i]) for i in range(b)]


def candidate_ranks(model, table, q1, q2, params, negative_sample, n_hard, err_flag=None, branches=1):
    """The other branch of test_step_mp (train_process.py:118-128, 141-147): the evaluation set brings its own
    candidates.  negative_sample [B, C] int64 on the table's device, -1 = padding; the first n_hard[b] candidates
    of query b are its hard answers (n_hard: sequence or int tensor of B counts).  Returns (negative_logit [B, C]
    with the -1e6 bias on the padding, ranking [B, C] int64, filtered ranks of the hard answers [B, max n_hard]
    int64, 0 in unused slots) -- one launch, no argsort.  branches > 1: union queries, q1/q2 [B, branches, dim],
    logits are the maximum over the branches."""
    if q1.numel() % (branches * q1.shape[-1]):
        raise _lib.SmxError("q1 must hold `branches` rows per query")
    b = q1.numel() // (branches * q1.shape[-1])
    if negative_sample.dim() != 2 or negative_sample.shape[0] != b or negative_sample.dtype != torch.int64:
        raise _lib.SmxError("negative_sample must be int64 [B, C]")
    dev = table.device
    cand = negative_sample.to(dev).contiguous()
    counts = _counts(n_hard)
    low, high = (int(x) for x in counts.aminmax()) if counts.numel() == b else (-1, 0)
    if low < 0 or high > cand.shape[1]:
        raise _lib.SmxError("one hard-answer count per query, between 0 and C")
    h = max(1, high)
    counts = _counts_on(counts, dev)
    q1c = q1.reshape(b * branches, -1).contiguous()
    q2c = None if q2 is None else q2.reshape(b * branches, -1).contiguous()
    _, _, dim = _dims(model, table, cand, q1c[:b], None if q2c is None else q2c[:b])
    c = cand.shape[1]
    logit = torch.empty((b, c), dtype=torch.float32, device=dev)
    ranking = torch.empty((b, c), dtype=torch.int64, device=dev)
    hard = torch.empty((b, h), dtype=torch.int64, device=dev)
    with _on(dev):
        _lib.call("smx_rank_candidates_union", MODELS[model], _stream(table), _ptr(table), table.shape[0], _ptr(q1c),
                  _ptr(q2c), b, branches, dim, ctypes.byref(params), _ptr(cand), c, _ptr(counts), h, _ptr(logit),
                  _ptr(ranking), _ptr(hard), _ptr(err_flag))
    return logit, ranking, hard


def ranking_metrics(hard_ranks):
    """MRR, HITS1/3/10 and HITS1max of one query from the filtered ranks of its hard answers
    (train_process.py:146-152); an empty tensor gives zeros, as the reference does for a query whose
    answer is not among the candidates."""
    if hard_ranks.numel() == 0:
        return dict(MRR=0.0, HITS1=0.0, HITS3=0.0, HITS10=0.0, HITS1max=0.0)
    r = hard_ranks.to(torch.float32)
    return dict(MRR=float((1.0 / r).mean()), HITS1=float((r <= 1).float().mean()), HITS3=float((r <= 3).float().mean()),
                HITS10=float((r <= 10).float().mean()), HITS1max=float(r.min() == 1))
