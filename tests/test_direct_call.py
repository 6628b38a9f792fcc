"""run()'s and quantize_hidden()'s direct call (nothing moved, copied or converted) against their
general path: which calls take it, and that both give the same bits."""
import importlib.util
import types

import numpy as np
import pytest
import torch

import __graft_entry__ as ge


@pytest.fixture(scope="module")
def moe():
    ge.load_package()
    from mlsys26_flashinfer_moe_amd import moe as m
    return m


def _cpu_args(moe, T=3, **change):
    fp8 = torch.float8_e4m3fn
    a = dict(routing_logits=torch.zeros(T, 256), routing_bias=torch.zeros(256),
             hidden_states=torch.zeros(T, 7168).to(fp8), hidden_states_scale=torch.ones(56, T),
             gemm1_weights=torch.empty(32, 4096, 7168, dtype=fp8, device="meta"),
             gemm1_weights_scale=torch.ones(32, 32, 56),
             gemm2_weights=torch.empty(32, 7168, 2048, dtype=fp8, device="meta"),
             gemm2_weights_scale=torch.ones(32, 56, 16), local_expert_offset=0, routed_scaling_factor=2.5,
             output=torch.zeros(T, 7168, dtype=torch.bfloat16), packed=None)
    a.update(change)
    return a


def test_struct_bytes_are_the_ctypes_struct(moe):
    from mlsys26_flashinfer_moe_amd import _lib
    values = [2**63 + 1, 2, 1, 4, 5, 6, 7, 8, 2**40, 2**20, -20, 2.5, 12, 1]
    a = _lib.MoeFp8Args()
    for (name, _), v in zip(_lib.MoeFp8Args._fields_, values):
        setattr(a, name, v)
    assert bytes(a) == moe._ARGS.pack(*values)


def test_the_current_stream_without_torchs_private_functions(moe, monkeypatch):
    for name in ("_cuda_getDevice", "_cuda_getCurrentRawStream"):
        monkeypatch.delattr(torch._C, name, raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: types.SimpleNamespace(cuda_stream=70 + device))
    spec = importlib.util.spec_from_file_location(moe.__name__ + "_again", moe.__file__)
    again = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(again)
    assert again._current_stream_id() == 73
    assert not again._run_direct(**_cpu_args(again))


def test_tensors_off_the_gpu_take_the_general_path(moe):
    assert not moe._run_direct(**_cpu_args(moe))
    assert not moe._run_direct(**_cpu_args(moe, T=0))
    assert not moe._quantize_direct(torch.zeros(2, 7168), torch.zeros(2, 7168).to(torch.float8_e4m3fn), torch.zeros(56, 2))


@pytest.mark.parametrize("name, message", [
    ("routing_logits", "routing_logits must be float32"), ("routing_bias", "routing_bias must be"),
    ("hidden_states", "hidden_states must be"), ("hidden_states_scale", "hidden_states_scale must be"),
    ("gemm1_weights", "gemm1_weights must be"), ("gemm2_weights_scale", "gemm2_weights_scale must be")])
def test_an_array_in_place_of_a_tensor_meets_the_contracts_assertion(moe, name, message):
    a = _cpu_args(moe, **{name: np.zeros((3, 256), dtype=np.float32)})
    del a["packed"]
    with pytest.raises(AssertionError, match=message):
        moe.run(**a)


def _off(t, elements):
    """A contiguous tensor with t's values whose data starts `elements` elements into its storage."""
    flat = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    v = flat[elements:].view(t.shape)
    v.copy_(t)
    return v


# name -> (change of the arguments, whether the direct call takes it)
FORMS = {
    "plain": (lambda a: {}, True),
    "f32 output": (lambda a: {"output": torch.empty_like(a["output"], dtype=torch.float32)}, True),
    "f16 bias": (lambda a: {"routing_bias": a["routing_bias"].half()}, True),
    "f32 bias": (lambda a: {"routing_bias": a["routing_bias"].float()}, True),
    "tensor scalars": (lambda a: {"local_expert_offset": torch.tensor(64), "routed_scaling_factor": torch.tensor(2.5)}, True),
    "f16 output": (lambda a: {"output": torch.empty_like(a["output"], dtype=torch.float16)}, False),
    "transposed scales": (lambda a: {"hidden_states_scale": a["hidden_states_scale"].t().contiguous().t()}, False),
    "strided logits": (lambda a: {"routing_logits": torch.cat([a["routing_logits"]] * 2, 1)[:, :256]}, False),
    "cpu logits": (lambda a: {"routing_logits": a["routing_logits"].cpu()}, False),
    "logits off by 4 bytes": (lambda a: {"routing_logits": _off(a["routing_logits"], 1)}, False),
    "hidden off by 8 bytes": (lambda a: {"hidden_states": _off(a["hidden_states"].view(torch.uint8), 8).view(torch.float8_e4m3fn)}, False),
    "bias off by 2 bytes": (lambda a: {"routing_bias": _off(a["routing_bias"], 1)}, False),
    "output off by 2 bytes": (lambda a: {"output": _off(a["output"], 1)}, False),
    "strided output": (lambda a: {"output": torch.empty(a["output"].shape[0], 2 * 7168, dtype=torch.bfloat16, device="cuda")[:, :7168]}, False),
    "bias as a row": (lambda a: {"routing_bias": a["routing_bias"].view(1, 256)}, False),
    "offset that wraps": (lambda a: {"local_expert_offset": 2**32 + 64}, False),
}


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 3, 65, 300])
def test_direct_call_gives_the_general_paths_bits(moe, T):
    from mlsys26_flashinfer_moe_amd import inputs
    dev = torch.device("cuda")
    logits, bias, hq, hs = inputs.make_activations(T, 31 + T, dev, 64, (0, 1, 2))
    w13, s13, w2, s2 = inputs.make_weights(77, dev)
    base = dict(routing_logits=logits, routing_bias=bias, hidden_states=hq, hidden_states_scale=hs, gemm1_weights=w13,
                gemm1_weights_scale=s13, gemm2_weights=w2, gemm2_weights_scale=s2, local_expert_offset=64,
                routed_scaling_factor=2.5, output=torch.empty(T, 7168, dtype=torch.bfloat16, device=dev))
    for name, (change, direct) in FORMS.items():
        if T == 1 and name in ("transposed scales", "strided logits", "strided output"):
            continue   # one row or column is contiguous whatever its stride
        a = dict(base, **change(base))
        want = torch.empty_like(a["output"])
        moe._run(**{**a, "output": want}, packed=moe._AUTO)
        a["output"].zero_()
        assert moe._run_direct(**a, packed=moe._AUTO) == direct, name
        moe.run(**a)
        assert torch.equal(a["output"], want), name
        assert float(want.float().abs().max()) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 17])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_direct_quantiser_gives_the_general_paths_bits(moe, T, dtype):
    x = torch.randn(T, 7168, device="cuda").to(dtype)
    want = moe._quantize(x, None, None)
    q, s = torch.empty_like(want[0]), torch.empty_like(want[1])
    for src, direct in ((x, True), (_off(x, 1), False)):
        q.zero_(), s.zero_()
        assert moe._quantize_direct(src, q, s) == direct
        moe.quantize_hidden(src, out=q, out_scale=s)
        assert torch.equal(q.view(torch.uint8), want[0].view(torch.uint8)) and torch.equal(s, want[1])
    assert not moe._quantize_direct(x, None, None)
    assert not moe._quantize_direct(_off(x, 1), object(), object())   # declined before the outputs are looked at
    assert not moe._quantize_direct(x, _off(q.view(torch.uint8), 1).view(torch.float8_e4m3fn), s)
