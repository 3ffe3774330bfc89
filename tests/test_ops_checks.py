"""Argument checks of the torch-facing ops that stand between a caller and a raw device write: a caller-supplied
`out` must be exactly what the kernels write (shape, dtype, contiguity, device), and routing tensors must have the
shapes the C code reads.  The CPU tests exercise the shared check on host tensors; the `gpu` tests call the ops."""
import pytest
import torch

from trellis_serve_amd import ops


def test_check_out_rejects_what_the_kernels_cannot_write():
    like = torch.empty((3, 256), dtype=torch.float16)
    ops._check_out(torch.empty((3, 256), dtype=torch.float16), (3, 256), like)
    ops._check_out(torch.empty((3, 256), dtype=torch.bfloat16), (3, 256), like)
    with pytest.raises(ValueError, match="shape"):
        ops._check_out(torch.empty((3, 128), dtype=torch.float16), (3, 256), like)
    with pytest.raises(ValueError, match="must be one of"):
        ops._check_out(torch.empty((3, 256), dtype=torch.float32), (3, 256), like)
    with pytest.raises(ValueError, match="must be one of"):
        ops._check_out(torch.empty((3, 256), dtype=torch.bfloat16), (3, 256), like, (torch.float16,))
    with pytest.raises(ValueError, match="contiguous"):
        ops._check_out(torch.empty((256, 3), dtype=torch.float16).t(), (3, 256), like)
    with pytest.raises(ValueError, match="is on"):
        ops._check_out(torch.empty((3, 256), dtype=torch.float16, device="meta"), (3, 256), like)


def _group(k, ns, K=3, dev="cuda"):
    g = torch.Generator().manual_seed(1)
    trs = [torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, generator=g).to(dev) for n in ns]
    suhs = [torch.ones(k, dtype=torch.float16, device=dev) for _ in ns]
    svhs = [torch.ones(n, dtype=torch.float16, device=dev) for n in ns]
    return trs, suhs, svhs


@pytest.mark.gpu
def test_ops_reject_bad_out_and_routing_before_launching():
    trs, suhs, svhs = _group(256, [128, 256])
    x = torch.randn((2, 256), dtype=torch.float16, device="cuda")
    for bad in (torch.empty((2, 256), dtype=torch.float16, device="cuda"),          # too narrow
                torch.empty((2, 384), dtype=torch.float32, device="cuda"),          # fp32
                torch.empty((384, 2), dtype=torch.float16, device="cuda").t()):     # not contiguous
        with pytest.raises(ValueError):
            ops.linear(x, trs, suhs, svhs, 1, out=bad)
        with pytest.raises(ValueError):
            ops.linear_prefill(x, trs, suhs, svhs, 1, out=bad)
    E, H, I = 4, 256, 128
    g = torch.Generator().manual_seed(2)
    experts = {}
    for proj, (k, n) in {"gate": (H, I), "up": (H, I), "down": (I, H)}.items():
        experts[f"{proj}_trellis"] = torch.randint(-32768, 32768, (E, k // 16, n // 16, 48), dtype=torch.int16,
                                                   generator=g).cuda()
        experts[f"{proj}_suh"] = torch.ones((E, k), dtype=torch.float16, device="cuda")
        experts[f"{proj}_svh"] = torch.ones((E, n), dtype=torch.float16, device="cuda")
    xm = torch.randn((3, H), dtype=torch.float16, device="cuda")
    ids = torch.zeros((3, 2), dtype=torch.int32, device="cuda")
    w = torch.full((3, 2), 0.5, device="cuda")
    with pytest.raises(ValueError, match="top_k"):
        ops.moe_forward(xm, ids, w[:, :1].contiguous(), experts, 1)      # weights of another shape
    with pytest.raises(ValueError, match="top_k"):
        ops.moe_forward(xm, ids[:2], w[:2], experts, 1)                  # fewer routing rows than tokens
    with pytest.raises(ValueError):
        ops.moe_forward(xm, ids, w, experts, 1, out=torch.empty((3, H), dtype=torch.float32, device="cuda"))


@pytest.mark.gpu
def test_linear_takes_every_form_of_its_rows():
    """The rows of x as one 2-D tensor, as a strided view, with more and with fewer dimensions, in fp32 and empty, give
    the same results in x's shape and dtype; tensors off the GPU are refused before anything is launched."""
    from trellis_serve_amd.runtime import ops as runtime_ops
    trs, suhs, svhs = _group(256, [128, 256])
    g = torch.Generator().manual_seed(4)
    for fn, rows in ((ops.linear, 6), (ops.linear_prefill, 6), (runtime_ops.linear, 6), (runtime_ops.linear, 90)):
        x = torch.randn((rows, 256), generator=g).half().cuda()
        y = fn(x, trs, suhs, svhs, 1)
        assert y.shape == (rows, 384) and y.dtype == torch.float16
        wide = torch.zeros((rows, 512), dtype=torch.float16, device="cuda")
        wide[:, :256] = x
        assert torch.equal(fn(wide[:, :256], trs, suhs, svhs, 1), y)
        assert torch.equal(fn(x.view(2, rows // 2, 256), trs, suhs, svhs, 1), y.view(2, rows // 2, 384))
        one = fn(x[0], trs, suhs, svhs, 1)
        assert one.shape == (384,) and torch.equal(one, fn(x[:1], trs, suhs, svhs, 1)[0])
        assert fn(x[:0], trs, suhs, svhs, 1).shape == (0, 384)
        if fn is runtime_ops.linear:
            y32 = fn(x.float().view(1, rows, 256), trs, suhs, svhs, 1)
            assert y32.dtype == torch.float32 and torch.equal(y32, y.float().view(1, rows, 384))
        else:
            with pytest.raises(ValueError):
                fn(x.cpu(), trs, suhs, svhs, 1)
    with pytest.raises(ValueError):
        ops.had_in_group(torch.ones((1, 256), dtype=torch.float16), torch.ones(256, dtype=torch.float16, device="cuda"),
                         torch.empty((1, 256), dtype=torch.float16, device="cuda"))


class _Calls:
    """A library whose size functions and launches record whether the tensors' device was current."""

    def __init__(self, seen, here):
        self.seen, self.here = seen, here

    def __getattr__(self, name):
        def call(*args):
            self.seen.append((name, self.here[-1]))
            return 4096 if name.endswith("_bytes") else 0
        return call


def test_sizes_and_launches_that_follow_the_cu_count_run_on_the_tensors_device(monkeypatch):
    """Past 32 rows a linear's workspace and plan follow the current device's CU count: with the tensors on device 1 and
    device 0 current, both the size and the call are taken with device 1 current (calls switch only when it is not)."""
    here, switched = [0], []

    class On:
        def __init__(self, device):
            self.index = ops._dev_index(device)

        def __enter__(self):
            switched.append(self.index)
            here.append(self.index)

        def __exit__(self, *a):
            here.pop()

    seen = []
    lib = _Calls(seen, here)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: here[-1])
    monkeypatch.setattr(torch.cuda, "device", On)
    monkeypatch.setattr(ops._lib, "load", lambda *a: lib)
    monkeypatch.setattr(ops, "_ws", lambda kind, dev: type("W", (), {"reserve": lambda self, dev, n: None})())
    monkeypatch.setattr(ops, "workspace", lambda dev, n, kind="linear": torch.empty(n, dtype=torch.uint8))
    monkeypatch.setattr(ops, "_stream", lambda dev: 0)
    monkeypatch.setattr(ops, "_dev_index", lambda dev: 1)
    arr = (ops._lib.Exl3Shard * 1)(ops._lib.Exl3Shard(1, 1, 1, 128))
    monkeypatch.setattr(ops, "_shards", lambda *a: (arr, 256, 3))
    monkeypatch.setattr(ops, "_check_trellis", lambda t: (256, 128, 3))
    monkeypatch.setattr(ops, "_half", lambda t, name: t)
    x = torch.zeros((65, 256), dtype=torch.float16)
    dev = torch.device("cuda", 1)

    def everything():
        ops.linear(x, [], [], [], 1)
        ops.linear_prefill(x, [], [], [], 1)
        ops.gemm_rotated(x, x, 1)
        ops.reserve_linear(dev, 40, 256, 128, 3)
        ops.reserve_prefill(dev, 40, 256, 128, 1)

    everything()
    assert {n for n, _ in seen} >= {"exl3_linear", "exl3_linear_prefill", "exl3_gemm_rotated",
                                    "exl3_linear_workspace_bytes", "exl3_prefill_workspace_bytes",
                                    "exl3_gemm_rotated_workspace_bytes"}
    assert all(current == 1 for _, current in seen), seen
    assert here == [0] and switched == [1] * 5
    here[:] = [1]
    everything()
    assert switched == [1] * 7   # the two reservations, at load
