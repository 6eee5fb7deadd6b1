"""The native launch calls (csrc/py_calls.cpp) and the asynchronous upload:
the checks they make on tensors, tables kept as compiled arrays, and passes
that the host queues without waiting."""
import numpy as np
import pytest

import cev_hip
from cev_hip import CevError, configs


def test_calls_check_tensors_before_any_launch(cev):
    import torch
    z = lambda *s, dt=torch.float32: torch.zeros(*s, dtype=dt)  # noqa: E731
    rot = type("R", (), dict(cos=z(4, 64), sin=z(4, 64), rotary_dim=128, n_pos=4))
    pos = z(2, dt=torch.int32)
    with pytest.raises(CevError, match="float16") as e:
        cev_hip.qknorm_rope(z(2, 2, 128, dt=torch.float16), z(2, 1, 128), z(128), z(128), pos, rot, 1e-6)
    assert e.value.code == -2
    with pytest.raises(CevError, match="contiguous") as e:
        cev_hip.qknorm_rope(z(2, 128, 2).transpose(1, 2), z(2, 1, 128), z(128), z(128), pos, rot, 1e-6)
    assert e.value.code == -2
    with pytest.raises(CevError, match="int32"):
        cev_hip.qknorm_rope(z(2, 2, 128), z(2, 1, 128), z(128), z(128), pos.long(), rot, 1e-6)
    with pytest.raises(CevError, match="share the dtype"):
        cev_hip.rms_norm(z(2, 64), z(64, dt=torch.bfloat16), 1e-6)
    with pytest.raises(CevError, match="row stride"):
        cev_hip.swiglu(z(2, 64), z(3, 64))
    with pytest.raises(CevError, match="in x's dtype"):
        cev_hip.linear(z(2, 64), z(4, 32))
    with pytest.raises(CevError, match="int32"):
        cev_hip.gather_rows(z(4, 8), z(2, dt=torch.int64))
    with pytest.raises(TypeError):
        cev_hip.gather_rows(z(4, 8), [0, 1], out=z(2, 8))


def test_errors_inside_a_call_are_raised(cev):
    """A tensor accessor that throws after the interpreter lock was let go
    raises like any other (it used to end the process)."""
    import torch
    stream = type("Stream", (), {"cuda_stream": 0})()
    x = torch.zeros(2, 64)
    with pytest.raises(IndexError):
        cev_hip.swiglu(x, x, out=torch.zeros(()), stream=stream)
    with pytest.raises(IndexError):
        cev_hip.gather_rows(x, out=torch.zeros(()), stream=stream)


def test_missing_operands_are_the_abis_to_refuse(cev):
    """None where only a pointer is passed on reaches the ABI's own check (a
    call without q heads has no w_q)."""
    import torch
    z = lambda *s, dt=torch.float32: torch.zeros(*s, dtype=dt)  # noqa: E731
    stream = type("Stream", (), {"cuda_stream": None})()
    rot = type("R", (), dict(cos=z(4, 64), sin=z(4, 64), rotary_dim=128, n_pos=4))
    with pytest.raises(CevError, match="null q") as e:
        cev_hip.qknorm_rope(z(2, 2, 128), z(2, 1, 128), None, z(128), z(2, dt=torch.int32), rot, 1e-6, stream=stream)
    assert e.value.code == -1
    layer = cev_hip.GatedDeltaNet(1, 2, 2, 4, dtype=torch.float32, device="cpu")
    with pytest.raises(CevError) as e:
        layer(z(1, 2, 1024), z(1, 2, 512), z(1, 2, 4), z(1, 2, 4), None, z(4), z(4), z(128), stream=stream)
    assert e.value.code == -1


def test_token_ids_out_of_range_are_refused():
    """A Python token id beyond int32 raises instead of wrapping around."""
    from cev_hip.qwen3 import _i32
    with pytest.raises(OverflowError):
        _i32([1, 2**40])
    assert _i32([1, 2]).dtype == np.int32 and _i32(np.array([3, 4], np.int64)).tolist() == [3, 4]


def test_the_library_builds_without_torch():
    """The default make target compiles no Python module and runs no Python."""
    import os
    import subprocess
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rust-cev_amd")
    run = subprocess.run(["make", "-n", "-B", "-C", pkg, "PYTHON=/nonexistent"], capture_output=True, text=True)
    assert run.returncode == 0 and "libcev_hip.so" in run.stdout
    assert "_cev_calls" not in run.stdout and "nonexistent" not in run.stderr


def test_tables_keep_their_blocks(cev):
    """A built table compiles from the builder's array; reading or replacing
    its block list makes the list the table."""
    tab, _, _ = cev_hip.BlockTable.from_plans([(10, 14, 10)], [(0, 3), (0, 5)])
    kept = cev_hip.BlockTable.from_plans([(10, 14, 10)], [(0, 3), (0, 5)])[0]
    assert len(tab) == 3 and np.array_equal(tab.to_dense_mask(), kept.to_dense_mask())
    assert [b.as_tuple() for b in tab.blocks] == [tab.array()[i].as_tuple() for i in range(3)]
    kept.array()[0].q_len = 99  # the caller's copy
    assert kept.array()[0].q_len != 99
    tab.blocks.pop()
    assert len(tab) == 2 and np.isneginf(tab.to_dense_mask()[-1]).all()


def test_plans_larger_than_the_first_guess(cev):
    """Many segments per row: the plan is built at its exact size."""
    n = 60
    blocks = [cev_hip.BlockTable.block(4 * i, 1, 400 + 4 * i, spans=[(100 * k, 20 + i) for k in range(4)]) for i in range(n)]
    tab = cev_hip.BlockTable(blocks, 4 * n, 400)
    plan = cev_hip.AttnPlan(cev_hip.attn_desc(cev_hip.CEV_BF16, 8, 8, 128, 4 * n, 400), tab)
    assert plan.nbytes == plan.host.nbytes == int(plan.header()[14]) and plan.n_tiles == n


@pytest.mark.gpu
def test_queued_passes_do_not_share_uploads(gpu):
    """Passes queued back to back, each with its own tables in flight, give
    what each gives alone."""
    import torch
    from cev_hip.qwen3 import Qwen3Stack
    w = configs.c2(bf16=True, n_layers=1, state_tokens=64, questions=4, q_len=20)
    g = torch.Generator(device=gpu).manual_seed(3)
    weights = {name: torch.randn(*shape, generator=g, device=gpu) * w.std for name, _, shape in w.weight_specs()}
    weights.update({name: torch.ones(n, device=gpu) for name, n in w.norm_specs()})
    stack = Qwen3Stack(w, weights, gpu, capacity=256)
    rng = np.random.default_rng(4)
    stack.prefill(0, rng.integers(0, w.vocab, 64), 512)
    passes = []
    for i in range(8):
        tab, pos, slots, gather = cev_hip.BlockTable.from_slots([(0, 64, 64)], [(0, 5 + i, 64), (0, 20 - i, 100)], 256)
        passes.append((rng.integers(0, w.vocab, tab.t), pos, slots, tab, gather))
    go = lambda p: stack.hidden(stack.run(*p[:4]), p[4])  # noqa: E731
    alone = []
    for p in passes:
        alone.append(go(p).clone())
        torch.cuda.synchronize()
    queued = [go(p) for p in passes]
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(alone, queued))
    with torch.cuda.graph(torch.cuda.CUDAGraph()), pytest.raises(RuntimeError, match="captured"):
        cev_hip.upload_async([np.zeros(4, np.int32)], gpu)
