"""The device deadline path, forced from the host (no wait is made to hang).

A runner whose deadline is one tick (10 ns) gives up every wait at once: the
routing reads part sums that have not landed (the unset marker, a NaN, so every
choice is -inf and the row picks experts 0 .. topk-1 with weight 0), the
hand-offs pass with their data half written, and the launch ends normally. Every
address a launch derives from hand-off data is clamped (expert ids to [0, E),
pick slots to the step's picks), and the picks that a workgroup polls take an
expert each in their row whatever it read, so that its table of them is whole:
a launch that gave up stays within its buffers. The tests assert the error words
(code, stage, workgroup, count), the table, and that ``clear_errors`` (a full workspace reset) restores a launch bit-identical
to a launch on a fresh workspace. The reference's guard test does the same
from its side (``test/kernels/test_guard_hip.py``, ``common/guard.py:69-89``).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit,experts,topk", [(0, 16, 4), (1, 256, 8), (7, 384, 6), (8, 384, 6)])
@pytest.mark.parametrize("rows", [1, 9, 33, 48])
def test_union_is_whole_whatever_was_read(unit, experts, topk, rows):
    """Picks as a wait that gave up may leave them (unset, a row half set with the experts that unset
    ones are clamped to, any words): every place of the union's order holds one pick, and a row's picks
    have an expert each. Valid picks keep theirs."""
    from sgl_amd_mono.moe import _lib

    g = torch.Generator().manual_seed(rows)
    valid = torch.stack([torch.randperm(experts, generator=g)[:topk] for _ in range(rows)]).to(torch.int32)
    valid[:, 0] = torch.where((valid == 0).any(1), valid[:, 0], 0)  # the expert that unset picks clamp to
    unset, half = torch.full_like(valid, -1), valid.clone()
    half[:, topk // 2 :] = -1
    words = torch.randint(-(2**31), 2**31 - 1, valid.shape, generator=g).to(torch.int32)
    last = torch.full_like(valid, experts - 1)
    for name, ids in (("valid", valid), ("unset", unset), ("half", half), ("words", words), ("last", last)):
        print(f"\nunit {unit} rows {rows}: {name}", flush=True)
        dev = ids.cuda()
        picks, got = torch.empty_like(dev), torch.empty_like(dev)
        rc = _lib.testing_lib().mkmoe_device_union(
            unit, rows, dev.data_ptr(), picks.data_ptr(), got.data_ptr(), torch.cuda.current_stream().cuda_stream
        )
        assert rc == 0
        got, order = got.cpu(), picks.flatten().cpu()
        assert bool((got >= 0).all()) and bool((got < experts).all()), name
        assert all(len(set(r)) == topk for r in got.tolist()), name
        assert order.tolist() == sorted(range(rows * topk), key=lambda t: (int(got.flatten()[t]), t)), name
        if name == "valid":
            assert torch.equal(got, ids)


@pytest.mark.parametrize(
    "workload,rows",
    [("cfg2_tp4_fp8", 8), ("cfg2_tp4_fp8", 24), ("cfg3_tp4_mxfp4", 8), ("cfg3_tp4_mxfp4", 24), ("cfg5_tp2_mxfp4_norm", 24)],
)
def test_deadline_gives_up_then_clear_restores(workload, rows):
    from test_gpu_parity import _case, _runner

    from sgl_amd_mono.moe import _lib

    c = _case(workload, rows)
    x = c.x[:rows].contiguous()
    ref_run = _runner(c)
    ref = ref_run.moe(c.w, x).clone()
    torch.cuda.synchronize()
    ref_run.raise_on_device_error()

    print(f"\n{workload} R={rows}: a launch with a one-tick deadline", flush=True)
    run = _runner(c, deadline_s=1e-8)
    out = run.moe(c.w, x)
    torch.cuda.synchronize()
    e = run.read_errors()
    print(f"  error words {e}", flush=True)
    assert e[_lib.ERRW_CODE] == 1, e  # MKMOE_DEVERR_DEADLINE
    assert e[_lib.ERRW_STAGE] in _lib.STAGES, e
    assert 0 <= e[_lib.ERRW_BLOCK] < 256, e
    # one record a wave a wait at most: 8 waves x 256 workgroups x (3 waits + the routing poll)
    assert 1 <= e[_lib.ERRW_COUNT] <= 8 * 256 * 4, e
    with pytest.raises(RuntimeError, match="deadline"):
        run.raise_on_device_error()
    assert out.shape == ref.shape

    # the reset restores the workspace; the next launch equals the fresh workspace's bit for bit
    run.deadline_s = 2.0
    run.clear_errors()
    assert run.read_errors() == [0] * _lib.ERRW_WORDS
    out2 = run.moe(c.w, x)
    torch.cuda.synchronize()
    run.raise_on_device_error()
    assert torch.equal(out2.view(torch.int16), ref.view(torch.int16)), "launch after clear_errors"
    assert bool((run.region("router_parts_polled") == 0xFF).all()), "polled part sums left unset"


@pytest.mark.parametrize(
    "workload,rows,stage,wg",
    [
        ("cfg2_tp4_fp8", 8, 4, 5),  # the gate_up hand-off (C)
        ("cfg2_tp4_fp8", 24, 3, 17),  # the polled picks (above 8 rows)
        ("cfg3_tp4_mxfp4", 16, 6, 200),  # stage Q's hand-off
        ("cfg3_tp4_mxfp4", 1, 2, 0),  # the polled router part sums and the x codes
        ("cfg3_tp4_mxfp4", 1, 3, 10),  # the polled picks (a workgroup of the early shared gate_up)
        ("cfg2_tp4_fp8", 4, 3, 200),  # the shared intermediate, before the shared down
        ("cfg5_tp2_mxfp4_norm", 24, 1, 255),  # the RMSNorm's hand-off (above 16 rows: below, none)
    ],
)
def test_fault_injection_stalls_one_wait(workload, rows, stage, wg):
    """A wait stalled by the test fault injection (one workgroup, one stage: the reference's
    SGLANG_AMD_MONO_FAULT_INJECT, common/guard.py:69-89) runs to its deadline: the error words
    name that wait (its stage and workgroup, the fault word set; the waits it holds up may reach
    their deadlines first), the launch ends, and clear_errors restores a launch bit-identical to
    a fresh workspace's."""
    from test_gpu_parity import _case, _runner

    from sgl_amd_mono.moe import _lib

    c = _case(workload, rows)
    x = c.x[:rows].contiguous()
    ref_run = _runner(c)
    ref = ref_run.moe(c.w, x).clone()
    torch.cuda.synchronize()
    ref_run.raise_on_device_error()
    assert ref_run.read_errors() == [0] * _lib.ERRW_WORDS

    print(f"\n{workload} R={rows}: workgroup {wg}'s wait at stage {stage} stalled (deadline 1 ms)", flush=True)
    run = _runner(c, deadline_s=1e-3)
    run.moe(c.w, x, fault=(stage, wg))
    torch.cuda.synchronize()
    e = run.read_errors()
    print(f"  error words {e}", flush=True)
    assert e[_lib.ERRW_CODE] == 1, e  # MKMOE_DEVERR_DEADLINE
    assert e[_lib.ERRW_FAULT] == 1, e
    assert (e[_lib.ERRW_STAGE], e[_lib.ERRW_BLOCK]) == (stage, wg), e
    assert e[_lib.ERRW_COUNT] >= 1, e

    run.deadline_s = 2.0
    run.clear_errors()
    assert run.read_errors() == [0] * _lib.ERRW_WORDS
    out2 = run.moe(c.w, x)
    torch.cuda.synchronize()
    run.raise_on_device_error()
    assert torch.equal(out2.view(torch.int16), ref.view(torch.int16)), "launch after clear_errors"


@pytest.mark.parametrize("preset,layout,rows", [("dsv3_tp4_fp8", "row_major", 4), ("v41_tp2", "aiter", 1)])
def test_flags_stay_set_while_a_workgroup_still_reads_them(preset, layout, rows):
    """Below stage Q's rows a workgroup waits at B (the shared intermediate) after its own arrival at
    C, so the others may pass C, finish and leave while it still reads the B flags: they must stay set
    until the last workgroup is out. One workgroup's B wait is held for half a second; meanwhile,
    with the 255 others out, another stream copies the control words to the host."""
    import time

    from bench import make_layer
    from sgl_amd_mono.moe.presets import PRESETS
    from sgl_amd_mono.moe.runner import MoeRunner

    p = PRESETS[preset]
    g = torch.Generator(device="cuda").manual_seed(31)
    w = make_layer(p, g, "cuda", 0.0)
    x = torch.randn(rows, p.hidden, generator=g, device="cuda").to(torch.bfloat16)
    run = MoeRunner(p, layout=layout, deadline_s=0.5)
    ref = run.moe(w, x).clone()
    run.raise_on_device_error()
    # the control words: the exit count at word 5, from byte 256 the flag arrays N, A, B, C, Q of 256 words
    words = 64 + 5 * 256
    host = torch.empty(words, dtype=torch.int32, pin_memory=True)
    wg = 200  # routes the step itself (the early shared gate_up is on workgroups 0 .. 63 and 0 .. 143)
    for side in [torch.cuda.Stream() for _ in range(4)]:
        print(f"\n{preset} R={rows}: workgroup {wg} held at B", flush=True)
        done = torch.cuda.Event()
        run.moe(w, x, fault=(3, wg))
        done.record()
        time.sleep(0.1)
        with torch.cuda.stream(side):
            host.copy_(run.ws.view(torch.int32)[:words], non_blocking=True)
        side.synchronize()
        during = not done.query()  # (a stream on the launch's own hardware queue copies after it)
        torch.cuda.synchronize()
        e = run.read_errors()
        run.clear_errors()
        assert (e[1], e[2], e[4]) == (3, wg, 1), e
        if during:
            break
    else:
        pytest.fail("every copy waited for the launch")
    assert int(host[5]) == 255, "the other workgroups are out"
    n = {"dsv3_tp4_fp8": 64, "v41_tp2": 144}[preset]
    b = host[64 + 2 * 256 : 64 + 3 * 256]
    assert bool((b[:n] == 1).all()) and not bool(b[n:].any()), "the B flags"
    out = run.moe(w, x)
    run.raise_on_device_error()
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    assert not bool(run.ws.view(torch.int32)[:words].any()), "the control words are clear between launches"


@pytest.mark.parametrize("rows", [1, 8, 24])
def test_a_nan_scale_is_no_unset_pick(rows):
    """Routing weights that are the NaN of all ones (the caller's scale with those bits, carried through
    the product) are set picks to the workgroups that poll them: the launch ends without a deadline,
    with the staged launch's output, whose stages read the weights behind each other."""
    import ctypes

    from test_gpu_parity import _case, _runner

    from sgl_amd_mono.moe import _lib

    c = _case("cfg2_tp4_fp8", 24)
    x = c.x[:rows].contiguous()
    run = _runner(c, deadline_s=0.05)
    at = ctypes.addressof(run.shape) + _lib.Shape.routed_scale.offset
    ctypes.memmove(at, b"\xff" * 4, 4)
    wts = torch.zeros(rows, c.preset.topk, device="cuda")
    out = run.moe(c.w, x, topk_w=wts)
    run.raise_on_device_error()
    print(f"\nR={rows}: weights' bits {sorted({hex(v & 0xFFFFFFFF) for v in wts.view(torch.int32).flatten().tolist()})}")
    staged = run.moe(c.w, x, staged=True)
    assert torch.equal(out.view(torch.int16), staged.view(torch.int16))
    assert bool((run.region("picks_polled") == 0xFF).all())
