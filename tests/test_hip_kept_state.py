"""ma_fwd_keep / ma_bwd_kept through the operator: a recorded forward call keeps the states of its steps and its
backward reads them.  Same kernels on the same states, so the gradients equal those of ma_bwd, which runs the steps
again, bit for bit, and the output equals the unrecorded call's."""
import pytest
import torch

from helpers import DT, block_safe_mask, keep_kernel, seeded_qkv
from ma.ma_hip import monarch_attention_hip, monarch_attention_hip_backward

pytestmark = pytest.mark.gpu
DEV = "cuda"

CHAIN, SLICES = "chain_fwd_mfma", "resident_slice_mfma"
CASES = [  # E, H, N, D, B, T, pre, dtype, variant, masked, the kernel that records: rows per slot that do and do not fill a slot's 128-row grid
    (1, 1, 64, 32, 8, 1, False, "f16", None, False, CHAIN),        # one step: no aR slot
    (2, 3, 197, 64, 14, 3, True, "f16", None, True, SLICES),        # ragged, three steps
    (1, 8, 300, 72, 20, 2, False, "bf16", "chained", True, CHAIN),
    (1, 2, 1000, 64, 128, 3, True, "bf16", "staged", False, "r_step_pair"),
    (1, 2, 256, 48, 16, 2, False, "f32", None, True, "r_step_f32"),
    (1, 2, 45, 20, 8, 2, True, "f16", "generic", False, "r_step_kernel"),
    (1, 9, 512, 64, 32, 2, False, "f16", "resident", False, None),  # keeps nothing: the backward runs the steps again
    (16, 12, 512, 64, 32, 2, True, "bf16", None, True, CHAIN),      # the slice-resident kernel is not far enough ahead here
    # calls that the slice-resident kernel records (its strips both ways, waves and column classes; masked, padded, one step to three)
    (48, 16, 197, 64, 14, 3, True, "f16", None, False, SLICES), (24, 16, 256, 64, 16, 1, False, "bf16", None, True, SLICES),
    (13, 1, 60, 32, 19, 3, False, "f16", None, True, SLICES), (50, 1, 21, 80, 9, 3, True, "bf16", None, False, SLICES), (13, 1, 81, 48, 24, 3, True, "f16", None, True, SLICES),
    (67, 7, 53, 72, 7, 3, False, "f16", None, True, SLICES), (80, 1, 2100, 32, 47, 3, True, "bf16", None, False, SLICES), (79, 1, 2570, 32, 48, 2, False, "bf16", None, True, SLICES),
    (122, 1, 548, 64, 23, 3, False, "f16", None, True, SLICES), (26, 1, 221, 32, 56, 3, True, "f16", None, True, SLICES), (39, 13, 542, 32, 12, 3, True, "bf16", None, True, SLICES),
    # the chained kernel in four waves of up to two strips: five strips both ways, four and five, seven and six
    (1, 3, 5003, 128, 72, 2, True, "bf16", "chained", True, CHAIN), (1, 2, 60 * 70, 64, 60, 3, False, "f16", "chained", True, CHAIN), (1, 2, 9000, 72, 100, 2, False, "f16", "chained", False, CHAIN),
    # ... in eight waves, where one side has seven or eight strips and the other up to five, and in three, for blocks of three strips
    (1, 3, 2393, 72, 120, 2, True, "bf16", "chained", True, CHAIN), (1, 2, 2310, 80, 20, 3, False, "f16", "chained", True, CHAIN), (1, 2, 509, 64, 128, 2, True, "f16", "chained", False, CHAIN),
    (1, 2, 70 * 110, 128, 110, 2, False, "bf16", "chained", True, CHAIN), (1, 3, 1590, 64, 40, 3, True, "bf16", "chained", True, CHAIN),
    (2, 4, 236, 32, 40, 2, False, "f16", "chained", True, CHAIN), (1, 5, 470, 128, 47, 2, True, "bf16", "chained", False, CHAIN),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_kept_states_give_the_gradients_of_a_recomputation(case):
    E, H, N, D, B, T, pre, dt, variant, masked, kernel = CASES[case]
    q, k, v = (t.to(DEV) for t in seeded_qkv(E, H, N, D, DT[dt], seed=case))
    mask = block_safe_mask(E, N, B, seed=case).to(DEV) if masked else None
    assert kernel is None or keep_kernel(q, k, v, mask, T, B, pre, variant) == kernel
    w = torch.randn(v.shape, generator=torch.Generator().manual_seed(case)).to(DEV).to(v.dtype)
    bwd = variant if variant in ("staged", "generic") else None
    want = monarch_attention_hip_backward(q, k, v, mask, w, T, B, pre, variant=bwd)
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    out = monarch_attention_hip(*leaves, mask, T, B, pre, variant=variant)
    plain = monarch_attention_hip(q, k, v, mask, T, B, pre, variant=variant or ("auto" if dt == "f32" else "staged"))
    for _ in range(2):   # the kept state is only read: a second backward gives the same
        got = torch.autograd.grad(out, leaves, w, retain_graph=True)
        for name, a, b in zip("qkv", got, want):
            assert torch.equal(a, b), f"d{name}"
    assert torch.equal(out.detach(), plain)
    torch.autograd.grad(out, leaves, w)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, leaves, w)


def test_kept_state_goes_through_saved_tensor_hooks():
    """Activation checkpointing keeps nothing of the operator's own, save_on_cpu moves the state with the inputs, and a hook
    that returns it at another address or as a strided view is served; the gradients are the same bits."""
    from torch.autograd.graph import save_on_cpu, saved_tensors_hooks
    from torch.utils.checkpoint import checkpoint

    E, H, N, D, B, T = 2, 4, 500, 64, 32, 2
    leaves = [t.to(DEV).requires_grad_() for t in seeded_qkv(E, H, N, D, torch.float16)]
    mask = block_safe_mask(E, N, B).to(DEV)
    w = torch.randn(E, H, N, D, generator=torch.Generator().manual_seed(1)).to(DEV).half()

    def op(*x):
        return monarch_attention_hip(*x, mask, T, B, False)

    want = torch.autograd.grad(op(*leaves), leaves, w)
    seen = []

    def spread(t):   # every second byte of a larger buffer, one byte off
        seen.append(t.numel() * t.element_size())
        if t.dtype != torch.uint8:
            return t
        buf = torch.zeros(2 * t.numel() + 1, dtype=t.dtype, device=t.device)[1::2]
        return buf.copy_(t)

    with saved_tensors_hooks(spread, lambda t: t):
        out = op(*leaves)
    assert len(seen) == 5 and max(seen) > 4 * w.numel() * 2   # q, k, v, mask; 2 aL, aR, Y and the column sums
    for a, b in zip(torch.autograd.grad(out, leaves, w), want):
        assert torch.equal(a, b)
    with save_on_cpu():
        out = op(*leaves)
    for a, b in zip(torch.autograd.grad(out, leaves, w), want):
        assert torch.equal(a, b)

    op(*leaves)   # (the workspace is there)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = checkpoint(op, *leaves, use_reentrant=False)
    assert torch.cuda.memory_allocated() - before <= 2 * w.numel() * 2   # the output
    for a, b in zip(torch.autograd.grad(out, leaves, w), want):
        assert torch.equal(a, b)

    with saved_tensors_hooks(lambda t: t[:-1] if t.dtype == torch.uint8 else t, lambda t: t):
        out = op(*leaves)
    with pytest.raises(RuntimeError, match="saved-tensor hooks"):
        torch.autograd.grad(out, leaves, w)


@pytest.mark.parametrize("E,H,N,D,B,dt", [(16, 12, 512, 64, 32, "bf16"), (64, 12, 197, 64, 14, "f16"), (8, 8, 197, 64, 16, "f32")])
def test_a_recorded_call_that_keeps_no_state_runs_as_an_unrecorded_one(E, H, N, D, B, dt):
    """AUTO resolves these to the resident kernels, which keep no state in memory."""
    leaves = [t.to(DEV).requires_grad_() for t in seeded_qkv(E, H, N, D, DT[dt])]
    w = torch.ones_like(leaves[2])
    with torch.no_grad():
        plain = monarch_attention_hip(*leaves, None, 2, B, False)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = monarch_attention_hip(*leaves, None, 2, B, False, keep_state=False)
    assert torch.cuda.memory_allocated() - before <= w.numel() * w.element_size() + 512
    assert torch.equal(out.detach(), plain)
    want = monarch_attention_hip_backward(*leaves, None, w, 2, B, False)
    for a, b in zip(torch.autograd.grad(out, leaves, w), want):
        assert torch.equal(a, b)


def test_calls_release_the_gil():
    """A call that blocks on a full queue must not hold up other Python threads.  With a switch interval longer than the test
    a waiting thread runs only if the call lets it."""
    import sys
    import threading

    q, k, v = (t.to(DEV) for t in seeded_qkv(1, 2, 64, 32, torch.float16))
    monarch_attention_hip(q, k, v, None, 2, 8, False)
    ran, gate = [], threading.Lock()
    gate.acquire()

    def other():
        gate.acquire()
        ran.append(True)

    thread = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    try:
        thread.start()
        sys.setswitchinterval(1000.0)
        gate.release()
        for _ in range(2000):
            monarch_attention_hip(q, k, v, None, 2, 8, False)
            if ran:
                break
        done = bool(ran)
    finally:
        sys.setswitchinterval(interval)
        thread.join()
    assert done


def test_threads_on_one_stream_share_the_workspace():
    """Calls of several launches that read each other's state arrays, from several threads, all on the default stream."""
    import threading

    shapes = [(2, 4, 300, 64, 20, 3), (1, 8, 1000, 64, 130, 2), (1, 3, 500, 32, 16, 2), (2, 2, 700, 96, 72, 3)]
    problems = []
    for i, (E, H, N, D, B, T) in enumerate(shapes):
        x = [t.to(DEV) for t in seeded_qkv(E, H, N, D, torch.bfloat16, seed=i)]
        problems.append((x, T, B, monarch_attention_hip(*x, None, T, B, False, variant="staged")))
    wrong = []

    def work(i):
        x, T, B, want = problems[i % len(problems)]
        outs = [monarch_attention_hip(*x, None, T, B, False, variant="staged") for _ in range(100)]
        wrong.extend(i for o in outs if not torch.equal(o, want))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_matrix_call_leaves_the_cached_workspace_as_it_is():
    from ma import ma_hip

    ma_hip.clear_workspace_cache()
    q, k, v = (t.to(DEV) for t in seeded_qkv(1, 12, 1024, 64, torch.float16))
    monarch_attention_hip(q, k, v, None, 2, 256, False)
    sizes = [b.numel() for b in ma_hip._HOST.workspaces()]
    ma_hip.monarch_matrix_hip(q, k, None, 2, 256, False)
    assert [b.numel() for b in ma_hip._HOST.workspaces()] == sizes
