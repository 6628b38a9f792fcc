"""GEMM1 with 128-row items at the sizes where its last round of units is split into half tiles.

On 256 CUs the per-XCD list of n items holds 2n units for 32 work-groups, so that n items leave 2n % 32
units for the last round, split when at most 16: n = 1 and 8 (halves only, 2 and 16 units), 9
(18: whole), 16 (full rounds), 17 and 24 (one full round, then 2 and 16), 25 (18: whole), 33 (two
rounds, then 2). Experts come by descending item rows, so that the last round holds the smallest
items; lists of equal items bring the large ones there. The items have 1 to 128 rows around the 16-
and 32-row groups, on given top-k lists. The intermediate and the second half are held to the same
bounds as everywhere (one fp8 step, one bf16 step) at the first and last row of every split item, and
the split items' intermediate to the bytes that whole tiles give."""
import numpy as np
import pytest
import torch

import test_gpu_layer as tl
from oracle import dispatch as odsp
from oracle import layer as olayer

pytestmark = pytest.mark.gpu

T = 512
ROWS = (1, 15, 16, 17, 31, 32, 33, 64, 65, 96, 127, 128)


def _expert_rows(n_items, rows=None):
    """The experts' row counts: n_items items of `rows` rows, or of the counts above (33: the first
    expert has two items)."""
    counts = [rows or ROWS[i % len(ROWS)] for i in range(n_items)]
    return counts if n_items <= 32 else [2 * (rows or 128)] + counts[2:]


def _lists(expert_rows, rng):
    """Top-k lists with these local assignments."""
    ids = rng.integers(32, 256, (T, 8)).astype(np.int32)
    used = np.zeros(T, dtype=int)
    for e, rows in enumerate(expert_rows):
        order = np.lexsort((rng.random(T), used))[:rows]
        ids[order, used[order]] = e
        used[order] += 1
    return ids, (rng.random((T, 8)) * 0.5 + 0.1).astype(np.float32)


def _split_items(ids, tw):
    """The items whose units are split: the last of the list, experts by descending rows of an item."""
    d = odsp.dispatch(ids, tw, 0)
    items = odsp.work_items(d["expert_count"], d["expert_start"], 128)
    first = {}
    for e, _, rows, _ in items:
        first.setdefault(int(e), int(rows))
    order = sorted(range(len(items)), key=lambda i: (-first[int(items[i][0])], i))
    last = 2 * len(items) % 32
    return d, items, [items[i] for i in order[len(items) - last // 2:]] if last <= 16 else []


def _run(ids, tw, seed):
    gh = tl._gh()
    dev = torch.device("cuda:0")
    assert torch.cuda.get_device_properties(dev).multi_processor_count == 256
    w, _ = tl._weights()
    logits, bias, hq, hs = gh.inputs.make_activations(T, seed, dev)
    kw = dict(routing_logits=logits, routing_bias=bias, hidden_states=hq, hidden_states_scale=hs,
              gemm1_weights=w[0], gemm1_weights_scale=w[1], gemm2_weights=w[2], gemm2_weights_scale=w[3],
              local_expert_offset=0, routed_scaling_factor=2.5)
    out = torch.full((T, 7168), float("nan"), dtype=torch.bfloat16, device=dev)
    ws = gh.new_workspace(T, dev)
    gh.write(ws, "topk_ids", ids)
    gh.write(ws, "topk_weights", tw)
    args = gh.make_args(**kw, output=out)
    gh.route_dispatch(args, ws, skip_routing=1)
    gh.gemm1(args, ws)
    gh.gemm2_combine(args, ws)
    torch.cuda.synchronize()
    return kw, ws, out.float().cpu().numpy()


@pytest.mark.parametrize("n_items, rows", [(1, None), (8, None), (9, None), (16, None), (17, None), (24, None), (25, None),
                                           (33, None), (1, 65), (4, 96), (17, 97), (24, 128), (33, 113)])
def test_items_around_the_split_of_the_last_round(n_items, rows):
    rng = np.random.default_rng(n_items + (rows or 0))
    ids, tw = _lists(_expert_rows(n_items, rows), rng)
    print(f"{n_items} items of {rows or 'various'} rows", flush=True)
    d, items, split = _split_items(ids, tw)
    assert len(items) == n_items and len(split) == (2 * n_items % 32 // 2 if 2 * n_items % 32 <= 16 else 0)
    kw, ws, got = _run(ids, tw, 4000 + n_items)
    gh = tl._gh()
    assert gh.counters(ws)[0] == n_items
    local = np.flatnonzero((ids < 32).any(axis=1))
    assert np.all(np.isfinite(got[local]))
    assert np.all(got[np.sum(ids < 32, axis=1) == 0] == 0)
    npkw = gh.to_numpy_inputs({**kw, "gemm1_weights": kw["gemm1_weights"][:1], "gemm2_weights": kw["gemm2_weights"][:1]})
    _, wnp = tl._weights()
    npkw["gemm1_weights"], npkw["gemm1_weights_scale"], npkw["gemm2_weights"], npkw["gemm2_weights_scale"] = wnp
    npkw["dequant_cache"] = tl._WEIGHTS["cache"]
    ends = [d["sorted_token"][r] for _, r0, n, _ in split for r in (r0, r0 + n - 1)]
    tokens = np.unique(np.concatenate([np.array(ends, dtype=np.int64), rng.choice(local, min(8, len(local)), replace=False)]))
    emu = olayer.layer_forward(**npkw, mode="emulated", topk=(ids, tw), tokens=tokens, requant_block=tl._requant_block(T))
    act, sc = tl._read_act(ws, len(emu["sorted_slot"]))
    tl._check_intermediate(act, sc, emu, tl._wanted_rows(emu, tokens), f"{n_items} items")
    tl._check_second_half(got[tokens], npkw, act, sc, tokens, f"{n_items} items", topk=(ids, tw))


@pytest.mark.parametrize("expert_rows", [(1, 15, 16, 17, 31, 32, 33, 48), (64, 65, 80, 81, 96, 97, 127, 128), (112,) * 8])
def test_split_items_give_the_bytes_of_whole_tiles(expert_rows):
    """Eight items, all split, and the same ones with eight more: 32 units, one full round of whole tiles."""
    rng = np.random.default_rng(sum(expert_rows))
    ids, tw = _lists(expert_rows, rng)
    more = ids.copy()
    free = np.argwhere(ids >= 32)
    for e, pick in zip(range(8, 16), np.split(rng.permutation(len(free))[:8 * 40], 8)):
        more[tuple(free[pick].T)] = e
    assert len(_split_items(ids, tw)[2]) == 8 and not _split_items(more, tw)[2]
    n = sum(expert_rows)
    got = []
    for lists in (ids, more):
        print(f"{expert_rows} split {lists is ids}", flush=True)
        _, ws, _ = _run(lists, tw, 77)
        assert tl._gh().counters(ws)[0] == (8 if lists is ids else 16)
        got.append(tl._read_act(ws, n))   # experts 0 to 7 come first in either
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
