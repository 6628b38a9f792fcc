"""The smallest batches through moe_fp8_run and moe_fp8_run_packed, whose GEMM1 work-groups route the
tokens themselves (up to 4) on rings of their own depth (6 slots up to 2 tokens, 4 up to 4, packed 8), and whose
GEMM2 work-groups requantise GEMM1's rows (1 token, packed 2): the top-k lists against the oracle,
lists, dispatch and output bit for bit against the stage entry points, which route, dispatch and
requantise in launches of their own, and the requantised rows bit for bit against the formula and
the output against the same tokens in a larger batch, which requant_kernel requantises."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import routing as orouting

pytestmark = pytest.mark.gpu

_STATE = {}


def _weights():
    import gpu_helpers as gh
    if not _STATE:
        w = gh.inputs.make_weights(911, torch.device("cuda:0"))
        _STATE["w"], _STATE["p"] = w, gh.pkg.pack_weights(w[0], w[2])
    return gh, _STATE["w"], _STATE["p"]


def _call(gh, args, ws, packed, how="run"):
    lib = gh._lib.load()
    p, n = (packed.data_ptr(), packed.numel()) if packed is not None else (None, 0)
    if how == "stages":
        gh.route_dispatch(args, ws)
        gh.gemm1(args, ws)
        gh.gemm2_combine(args, ws)
    elif how == "profiled":
        events = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        for e in events:
            e.record()
        gh._lib.check(lib.moe_fp8_run_profiled(args, p, n, ws.ptr, ws.buffer.numel(), gh.stream(),
                                               (ctypes.c_void_p * 4)(*[e.cuda_event for e in events])), how)
    elif packed is not None:
        gh._lib.check(lib.moe_fp8_run_packed(args, p, n, ws.ptr, ws.buffer.numel(), gh.stream()), how)
    else:
        gh.run_layer(args, ws)


@pytest.mark.parametrize("bias_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 8, 9])
def test_small_batches(T, bias_dtype):
    gh, w, packed = _weights()
    dev = torch.device("cuda:0")
    print(f"T={T} bias {bias_dtype}", flush=True)
    for extreme in (False, True):
        logits, bias, hq, hs = gh.inputs.make_activations(T, 60 + T, dev, 32, (1, 7))
        if extreme:
            # ties, saturated scores, and a last token with five finite candidates
            logits = (logits * 4).round() * 30
            logits[-1] = float("-inf")
            logits[-1, 32:37] = torch.tensor([1.0, 2.0, 2.0, -1.0, 0.5], device=dev)
        bias = bias.to(bias_dtype)
        if extreme:
            bias = bias.float().masked_fill(torch.arange(256, device=dev) >= 40, float("-inf")).to(bias_dtype)
        want = None
        for pk, how in ((None, "stages"), (None, "run"), (None, "profiled"), (packed, "run"), (packed, "profiled")):
            out = torch.full((T, 7168), 7.0, dtype=torch.bfloat16, device=dev)
            ws = gh.new_workspace(T, dev)
            args = gh.make_args(logits, bias, hq, hs, w[0], w[1], w[2], w[3], 32, 2.5, out)
            for _ in range(2):
                _call(gh, args, ws, pk, how)
            torch.cuda.synchronize()
            ids = gh.read(ws, "topk_ids", torch.int32, T * 8).reshape(T, 8)
            tw = gh.read(ws, "topk_weights", torch.float32, T * 8).reshape(T, 8)
            gh.check_dispatch(ws, ids, tw, 32, T)
            got = (ids.tobytes(), tw.tobytes(), out.view(torch.int16).cpu().numpy().tobytes())
            want = want or got
            assert got == want, (T, extreme, pk is not None, how)
        oid, ow = orouting.route(logits.cpu().numpy(), bias.float().cpu().numpy(), 2.5)
        assert np.array_equal(ids, oid) and np.array_equal(tw.view(np.uint32), ow.view(np.uint32))


@pytest.mark.parametrize("boosted", [(), (1, 7), (1, 4, 7, 9, 12, 15, 20, 22)])
@pytest.mark.parametrize("T", [1, 2, 3])
def test_requantised_rows(T, boosted):
    gh, w, packed = _weights()
    dev = torch.device("cuda:0")
    big = 9
    logits, bias, hq, hs = gh.inputs.make_activations(big, 80, dev, 32, boosted)
    for pk in (None, packed):
        outs = []
        for n in (T, big):
            print(f"T={n} packed {pk is not None}", flush=True)
            out = torch.full((n, 7168), 7.0, dtype=torch.float32, device=dev)
            ws = gh.new_workspace(n, dev)
            args = gh.make_args(logits[:n].contiguous(), bias, hq[:n].contiguous(), hs[:, :n].contiguous(),
                                w[0], w[1], w[2], w[3], 32, 2.5, out)
            for _ in range(2):
                _call(gh, args, ws, pk)
            torch.cuda.synchronize()
            outs.append(out)
            rows = int(gh.read(ws, "counters", torch.int32, 2)[1])
            x = torch.from_numpy(gh.read(ws, "swiglu", torch.float32, rows * 2048).copy()).reshape(rows, 32, 64)
            scale = (x.abs().amax(-1) / 448.0).clamp_min(1e-12)
            q = (x / scale[..., None]).to(torch.float8_e4m3fn).view(torch.uint8).reshape(rows, 2048)
            assert rows > 0 or not boosted
            assert np.array_equal(gh.read(ws, "act", torch.uint8, rows * 2048).reshape(rows, 2048), q.numpy())
            assert np.array_equal(gh.read(ws, "act_scale", torch.float32, rows * 32).reshape(rows, 32), scale.numpy())
        assert torch.equal(outs[0], outs[1][:T])
