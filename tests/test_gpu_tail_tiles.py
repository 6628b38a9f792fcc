"""GEMM1 with 128-row items at the sizes where its last round of units is split into half tiles.

On 256 CUs the per-XCD list of n items holds 2n units for 32 work-groups, so that n items leave 2n % 32
units for the last round, split when at most 16: n = 1 and 8 (halves only, 2 and 16 units), 9
(18: whole), 16 (full rounds), 17 and 24 (one full round, then 2 and 16), 25 (18: whole), 33 (two
rounds, then 2). The items have 1 to 128 rows around the 16- and 32-row groups, on given top-k lists. The
intermediate and the second half are held to the same bounds as everywhere (one fp8 step, one
bf16 step)."""
import numpy as np
import pytest
import torch

import test_gpu_layer as tl
from oracle import layer as olayer

pytestmark = pytest.mark.gpu

ROWS = (1, 15, 16, 17, 31, 32, 33, 64, 65, 96, 127, 128)


def _lists(n_items, T, rng):
    """Top-k lists whose local assignments make n_items items of the row counts above (33: the
    first expert has two items)."""
    ids = rng.integers(32, 256, (T, 8)).astype(np.int32)
    used = np.zeros(T, dtype=int)
    for i in range(n_items):
        e = min(i, 31) if n_items <= 32 else max(i - 1, 0)
        rows = 128 if n_items > 32 and i < 2 else ROWS[i % len(ROWS)]
        order = np.lexsort((rng.random(T), used))[:rows]
        ids[order, used[order]] = e
        used[order] += 1
    return ids, (rng.random((T, 8)) * 0.5 + 0.1).astype(np.float32)


@pytest.mark.parametrize("n_items", [1, 8, 9, 16, 17, 24, 25, 33])
def test_items_around_the_split_of_the_last_round(n_items):
    gh = tl._gh()
    dev = torch.device("cuda:0")
    w, wnp = tl._weights()
    T = 512
    rng = np.random.default_rng(n_items)
    ids, tw = _lists(n_items, T, rng)
    print(f"{n_items} items", flush=True)
    logits, bias, hq, hs = gh.inputs.make_activations(T, 4000 + n_items, dev)
    kw = dict(routing_logits=logits, routing_bias=bias, hidden_states=hq, hidden_states_scale=hs,
              gemm1_weights=w[0], gemm1_weights_scale=w[1], gemm2_weights=w[2], gemm2_weights_scale=w[3],
              local_expert_offset=0, routed_scaling_factor=2.5)
    out = torch.full((T, 7168), float("nan"), dtype=torch.bfloat16, device=dev)
    ws = gh.new_workspace(T, dev)
    gh.write(ws, "topk_ids", ids)
    gh.write(ws, "topk_weights", tw)
    args = gh.make_args(**kw, output=out)
    gh.route_dispatch(args, ws, skip_routing=1)
    assert gh.counters(ws)[0] == n_items
    gh.gemm1(args, ws)
    gh.gemm2_combine(args, ws)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    npkw = gh.to_numpy_inputs({**kw, "gemm1_weights": w[0][:1], "gemm2_weights": w[2][:1]})
    npkw["gemm1_weights"], npkw["gemm1_weights_scale"], npkw["gemm2_weights"], npkw["gemm2_weights_scale"] = wnp
    npkw["dequant_cache"] = tl._WEIGHTS["cache"]
    local = np.flatnonzero((ids < 32).any(axis=1))
    tokens = np.sort(rng.choice(local, min(12, len(local)), replace=False))
    emu = olayer.layer_forward(**npkw, mode="emulated", topk=(ids, tw), tokens=tokens, requant_block=tl._requant_block(T))
    act, sc = tl._read_act(ws, len(emu["sorted_slot"]))
    tl._check_intermediate(act, sc, emu, tl._wanted_rows(emu, tokens), f"{n_items} items")
    tl._check_second_half(got[tokens], npkw, act, sc, tokens, f"{n_items} items", topk=(ids, tw))
    assert np.all(got[np.sum(ids < 32, axis=1) == 0] == 0)
