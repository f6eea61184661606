"""The declarative argument contracts (fusedtok_amd/_contract.py) and the
sampling-argument normalisation (fusedtok_amd/_sampling_args.py), on the
host: shape binding, messages, error classes, in-place staging rules and
the three history forms. No device is needed."""

import numpy as np
import pytest
import torch

import fusedtok_amd as ft
from fusedtok_amd import _contract as _contract_mod
from fusedtok_amd import _sampling_args as sa
from fusedtok_amd._contract import Arr, Contract, Idx, Rule


def test_symbols_bind_across_operands():
    c = Contract(Arr("q", "B Hq D"), Arr("k", "B Hkv T D", mismatch="k must match q"),
                 Idx("lens", "B", lambda c: c.T, optional=True, what="lens shape"))
    call = c.bind(q=np.zeros((2, 8, 16), np.float32), k=np.zeros((2, 4, 5, 16), np.float32),
                  lens=np.array([5, 0], np.int32))
    assert (call.B, call.Hq, call.Hkv, call.T, call.D) == (2, 8, 4, 5, 16)
    assert not call.on_gpu
    with pytest.raises(ValueError, match="k must match q"):
        c.bind(q=np.zeros((2, 8, 16), np.float32), k=np.zeros((2, 4, 5, 8), np.float32),
               lens=None)
    with pytest.raises(ValueError, match=r"lens entries must be in \[0, 5\]"):
        c.bind(q=np.zeros((2, 8, 16), np.float32), k=np.zeros((2, 4, 5, 16), np.float32),
               lens=np.array([6, 0]))
    with pytest.raises(ValueError, match="lens shape"):
        c.bind(q=np.zeros((2, 8, 16), np.float32), k=np.zeros((2, 4, 5, 16), np.float32),
               lens=np.array([1, 2, 3]))


def test_optional_leading_dim_and_same_shape():
    c = Contract(Arr("x", "rows? cols"), Arr("r", "=x", optional=True, mismatch="r vs x"))
    assert c.bind(x=np.zeros(7, np.float32), r=None).rows == 1
    assert c.bind(x=np.zeros((3, 7), np.float32), r=None).rows == 3
    with pytest.raises(ValueError, match="r vs x"):
        c.bind(x=np.zeros((3, 7), np.float32), r=np.zeros((7,), np.float32))


def test_open_bound_and_rules():
    c = Contract(Arr("cache", "B T"), Idx("lens", "B", lambda c: c.T, open_bound=True,
                                          what="w"),
                 rules=(Rule(lambda c: c.T % 2 == 0, "T must be even"),))
    with pytest.raises(ValueError, match=r"\[0, 4\)"):
        c.bind(cache=np.zeros((1, 4), np.float32), lens=[4])
    with pytest.raises(ValueError, match="T must be even"):
        c.bind(cache=np.zeros((1, 3), np.float32), lens=[0])
    with pytest.raises(TypeError, match="integer values"):
        c.bind(cache=np.zeros((1, 4), np.float32), lens=[0.5])


def test_inplace_host_operands_must_be_writable_float32():
    with pytest.raises(TypeError, match="in-place"):
        ft.kv_append(np.zeros((1, 1, 4, 4), np.float64), np.zeros((1, 1, 4, 4), np.float32),
                     np.zeros((1, 1, 4), np.float32), np.zeros((1, 1, 4), np.float32), [0])
    strided = np.zeros((1, 1, 4, 8), np.float32)[..., ::2]
    with pytest.raises(TypeError, match="in-place"):
        ft.kv_append(strided, strided.copy(), np.zeros((1, 1, 4), np.float32),
                     np.zeros((1, 1, 4), np.float32), [0])


def test_host_messages_of_the_public_ops():
    q = np.zeros((1, 4, 8), np.float32)
    k = np.zeros((1, 2, 6, 8), np.float32)
    with pytest.raises(ValueError, match="head counts"):
        ft.attention_decode(np.zeros((1, 0, 8), np.float32), k, k)
    with pytest.raises(ValueError, match="multiple of kv heads"):
        ft.attention_decode(np.zeros((1, 3, 8), np.float32), k, k)
    with pytest.raises(ValueError, match=r"q must be \[B, Hq, D\]"):
        ft.attention_decode(np.zeros((4, 8), np.float32), k, k)
    with pytest.raises(ValueError, match="multiple of 4 and at most 512"):
        ft.attention_decode(np.zeros((1, 2, 6), np.float32), np.zeros((1, 1, 3, 6), np.float32),
                            np.zeros((1, 1, 3, 6), np.float32))
    with pytest.raises(ValueError, match="block_table must be"):
        ft.attention_decode_paged(q, np.zeros((3, 2, 4, 8), np.float32),
                                  np.zeros((3, 2, 4, 8), np.float32), np.zeros((2, 1), np.int32))
    with pytest.raises(ValueError, match=r"block_table entries must be in \[0, 3\)"):
        ft.attention_decode_paged(q, np.zeros((3, 2, 4, 8), np.float32),
                                  np.zeros((3, 2, 4, 8), np.float32), np.array([[3]]))
    with pytest.raises(ValueError, match="even"):
        ft.rope(np.zeros((2, 5), np.float32))
    with pytest.raises(ValueError, match="pos_offset"):
        ft.rope(np.zeros((2, 4), np.float32), pos_offset=-2)
    with pytest.raises(TypeError, match="a_q"):
        ft.qgemm(np.ones((2, 4), np.float32), 0.5, np.ones((3, 4), np.int8), 0.5)
    with pytest.raises(TypeError, match="b_q"):
        ft.qgemm(np.ones((2, 4), np.int8), 0.5, np.ones((3, 4), np.float32), 0.5)
    with pytest.raises(TypeError, match="int8"):
        ft.dequantize_int8(np.ones(4, np.float32), 0.5)
    with pytest.raises(TypeError, match="GPU int8"):
        ft.qadd_int8(np.ones(4, np.int8), 0.5, np.ones(4, np.int8), 0.5)
    with pytest.raises(TypeError, match="no host path"):
        ft.rmsnorm_quant(np.ones((2, 4), np.float32), np.ones(4, np.float32))


def test_sampling_params_and_seeds():
    with pytest.raises(ValueError, match="p must be"):
        ft.sample_topp(np.zeros(4, np.float32), 0.0)
    with pytest.raises(ValueError, match="temperature"):
        ft.sample_topp(np.zeros(4, np.float32), 0.5, temperature=0.0)
    with pytest.raises(ValueError, match="penalty"):
        ft.decode_step(np.zeros(4, np.float32), [0], 0.0)
    with pytest.raises(ValueError, match="empty logits"):
        ft.sample_topp(np.zeros(0, np.float32), 0.5)
    np.testing.assert_array_equal(sa.seed_vector(None, 3), [0, 1, 2])
    np.testing.assert_array_equal(sa.seed_vector(np.array([2 ** 63 - 1], np.uint64), 1),
                                  [2 ** 63 - 1])
    with pytest.raises(ValueError, match=r"2\*\*63"):
        sa.seed_vector(np.array([2 ** 63], np.uint64), 1)
    with pytest.raises(ValueError, match=r"2\*\*63"):
        sa.seed_vector([-1], 1)
    with pytest.raises(TypeError, match="integers"):
        sa.seed_vector([0.5], 1)
    with pytest.raises(ValueError, match="one entry per row"):
        sa.seed_vector([1, 2], 3)
    with pytest.raises(ValueError, match="1-D"):
        sa.seed_vector([[1]], 1)


def test_history_forms_give_one_csr_layout():
    ragged = [[3, 1], [], [4, 4, 0]]
    flat, offs = sa.histories_csr(ragged, None, 3, 8)
    np.testing.assert_array_equal(flat, [3, 1, 4, 4, 0])
    np.testing.assert_array_equal(offs, [0, 2, 2, 5])
    f2, o2 = sa.histories_csr(np.array([3, 1, 4, 4, 0]), np.array([0, 2, 2, 5]), 3, 8)
    np.testing.assert_array_equal(f2, flat)
    np.testing.assert_array_equal(o2, offs)
    f3, o3 = sa.histories_csr(torch.tensor([[1, 2], [3, 4]]), None, 2, 8)
    np.testing.assert_array_equal(f3, [1, 2, 3, 4])
    np.testing.assert_array_equal(o3, [0, 2, 4])
    with pytest.raises(ValueError, match=r"\[0, 8\)"):
        sa.histories_csr([[8]], None, 1, 8)
    with pytest.raises(ValueError, match="non-decreasing"):
        sa.histories_csr(np.array([1, 2]), np.array([0, 2, 1]), 2, 8)
    with pytest.raises(TypeError, match="ids_offsets"):
        sa.histories_csr(np.array([1, 2]), np.array([0.0, 1.5, 2.0]), 2, 8)
    with pytest.raises(ValueError, match="one entry per row"):
        sa.histories_csr([[1]], None, 2, 8)
    np.testing.assert_array_equal(sa.history_1d([5, 0], 6, None), [5, 0])
    with pytest.raises(ValueError, match=r"\[0, 6\)"):
        sa.history_1d([6], 6, None)


class _DeviceTensor(torch.Tensor):
    """A CPU tensor that says it is on the GPU: bind only looks at it."""
    is_cuda = property(lambda self: True)


def _dev(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype).as_subclass(_DeviceTensor)


def _bind_by_the_general_routines(contract, values):
    """Contract.bind for device operands, every check through the general
    routine of its operand."""
    call = _contract_mod.Call(contract, dict(values), values[contract.operands[0].name].device)
    shapes = {}
    for spec in contract.operands:
        v = values.get(spec.name)
        if v is None:
            if not spec.optional:
                raise TypeError(f"{spec.name} is required")
            continue
        if isinstance(spec, Arr):
            v = spec.on_device(v)
            if spec.same_dtype is not None:
                if v.dtype is not getattr(call, spec.same_dtype).dtype:
                    raise TypeError(f"{spec.name} must have the same dtype as {spec.same_dtype}")
            contract._bind_shape(call, spec, tuple(v.shape), shapes)
        else:
            v = contract._index(call, spec, v, True, shapes)
        setattr(call, spec.name, v)
    for rule in contract.rules:
        if not rule.test(call):
            raise rule.exc(rule.message)
    return call


_HALF = torch.bfloat16
_PAGED = dict(q=_dev(2, 8, 64), k_pool=_dev(9, 2, 16, 64), v_pool=_dev(9, 2, 16, 64),
              block_table=_dev(2, 4, dtype=torch.int32), lens=_dev(2, dtype=torch.int32))
_NORM = dict(x=_dev(3, 8), weight=_dev(8), residual=_dev(3, 8))


@pytest.mark.parametrize("contract,base,change", [
    ("_DECODE_PAGED", _PAGED, {}),
    ("_DECODE_PAGED", _PAGED, dict(lens=None)),
    ("_DECODE_PAGED", _PAGED, dict(q=_dev(2, 8))),                      # rank
    ("_DECODE_PAGED", _PAGED, dict(k_pool=_dev(9, 2, 16, 32))),         # D differs
    ("_DECODE_PAGED", _PAGED, dict(v_pool=_dev(9, 2, 8, 64))),          # not k_pool's shape
    ("_DECODE_PAGED", _PAGED, dict(k_pool=_dev(9, 2, 16, 64, dtype=_HALF))),   # storage type
    ("_DECODE_PAGED", _PAGED, dict(q=_dev(2, 8, 64, dtype=torch.float64))),
    ("_DECODE_PAGED", _PAGED, dict(q=_dev(2, 64, 8).transpose(1, 2))),  # not contiguous
    ("_DECODE_PAGED", _PAGED, dict(k_pool=np.zeros((9, 2, 16, 64), np.float32))),
    ("_DECODE_PAGED", _PAGED, dict(k_pool=torch.zeros(9, 2, 16, 64))),  # a CPU tensor
    ("_DECODE_PAGED", _PAGED, dict(v_pool=None)),                       # required
    ("_DECODE_PAGED", _PAGED, dict(lens=_dev(3, dtype=torch.int32))),
    ("_DECODE_PAGED", _PAGED, dict(lens=_dev(2, dtype=torch.int64))),   # converted
    ("_DECODE_PAGED", _PAGED, dict(lens=[1, 2])),                       # uploaded
    ("_DECODE_PAGED", _PAGED, dict(lens=[1, 65])),                      # out of range
    ("_DECODE_PAGED", _PAGED, dict(lens=np.array([0.5, 1.0]))),
    ("_DECODE_PAGED", _PAGED, dict(block_table=_dev(8, dtype=torch.int32))),
    ("_DECODE_PAGED", _PAGED, dict(block_table=_dev(4, 2, dtype=torch.int32).t())),
    ("_DECODE_PAGED", _PAGED, dict(q=_dev(2, 6, 64))),                  # a rule: the group
    ("_RMSNORM", _NORM, {}),
    ("_RMSNORM", _NORM, dict(residual=None)),
    ("_RMSNORM", _NORM, dict(x=_dev(8), residual=_dev(8))),             # no leading dimension
    ("_RMSNORM", _NORM, dict(x=_dev(1, 3, 8))),
    ("_RMSNORM", _NORM, dict(residual=_dev(3, 4))),
    ("_RMSNORM", _NORM, dict(weight=_dev(9))),
    ("_RMSNORM", _NORM, dict(weight=_dev(8, dtype=_HALF))),             # converted
    ("_RMSNORM", _NORM, dict(weight=_dev(16)[::2])),                    # made contiguous
    ("_RMSNORM", _NORM, dict(x=_dev(3, 0), weight=_dev(0), residual=None)),  # a rule
])
def test_device_binding_equals_the_general_routines(contract, base, change):
    # bind's inline checks for device operands against the operands' general
    # routines, over every form they tell apart: the same symbols and
    # operands, or the same error
    contract = getattr(ft, contract)

    def outcome(bind):
        try:
            call = bind({**base, **change})
        except (TypeError, ValueError) as exc:
            return type(exc), str(exc)
        ops = {s.name: getattr(call, s.name) for s in contract.operands}
        return dict(call.dims), {k: None if v is None else (tuple(v.shape), v.dtype, v.is_contiguous())
                                 for k, v in ops.items()}, call.on_gpu

    got = outcome(lambda values: contract.bind(**values))
    assert got == outcome(lambda values: _bind_by_the_general_routines(contract, values))


@pytest.mark.parametrize("missing", ["_raw_stream", "_raw_device"])
def test_current_stream_without_torchs_raw_calls(missing, monkeypatch):
    class Stream:
        cuda_stream = 77

    monkeypatch.setattr(_contract_mod, missing, None)
    monkeypatch.setattr(torch.cuda, "current_stream", Stream)
    assert _contract_mod.current_stream() == 77


@pytest.mark.gpu
def test_current_stream_is_torchs():
    streams = [torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    for stream in streams + streams[:1]:
        with torch.cuda.stream(stream):
            assert _contract_mod.current_stream() == stream.cuda_stream
            assert stream.cuda_stream == torch.cuda.current_stream().cuda_stream
