"""Routing and dispatch around the sizes where the kernels change (one work-group up to 128 tokens, one
token per wavefront and quarter-block histograms up to 2048, 16-token blocks above): top-k lists and
dispatch arrays bit for bit against the oracle, from logits and from given lists."""
import numpy as np
import pytest
import torch

from oracle import routing as orouting

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [127, 128, 129, 131, 143, 144, 145, 255, 256, 257, 301, 1024, 2047, 2048, 2049])
def test_route_and_dispatch(T):
    import gpu_helpers as gh
    dev = torch.device("cuda:0")
    print(f"T={T}", flush=True)
    off = 64
    logits, bias, hq, hs = gh.inputs.make_activations(T, 300 + T, dev, off, (2, 30))
    logits[-1] = float("-inf")   # ties: one expert several times
    logits[-1, off:off + 3] = 1.0
    out = torch.empty((T, 7168), dtype=torch.bfloat16, device=dev)
    dummy = torch.zeros(16, dtype=torch.float32, device=dev)
    ws = gh.new_workspace(T, dev)
    args = gh.make_args(logits, bias, hq, hs, dummy, dummy, dummy, dummy, off, 2.5, out)
    oid, ow = orouting.route(logits.cpu().numpy(), bias.float().cpu().numpy(), 2.5)
    for _ in range(2):
        gh.route_dispatch(args, ws)
        ids = gh.read(ws, "topk_ids", torch.int32, T * 8).reshape(T, 8)
        w = gh.read(ws, "topk_weights", torch.float32, T * 8).reshape(T, 8)
        assert np.array_equal(ids, oid) and np.array_equal(w.view(np.uint32), ow.view(np.uint32))
        gh.check_dispatch(ws, ids, w, off, T)
    rng = np.random.default_rng(T)
    lists = {"random": rng.integers(-1, 256, (T, 8)), "one expert": np.full((T, 8), off + 31),
             "none local": np.full((T, 8), off - 1)}
    for name, ids in lists.items():
        print(f"T={T} {name}", flush=True)
        ids = ids.astype(np.int32)
        w = rng.random((T, 8), dtype=np.float32)
        gh.write(ws, "topk_ids", ids)
        gh.write(ws, "topk_weights", w)
        gh.route_dispatch(args, ws, skip_routing=1)
        gh.check_dispatch(ws, ids, w, off, T)
