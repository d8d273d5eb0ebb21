"""The native per-call path of the Python entry points (csrc/fast_calls.cpp).

It takes the common form of the arguments and leaves every other form to the
general path: same results, same conversions, same errors.
"""

from __future__ import annotations

import ctypes
import threading

import pytest
import torch

from aws_training_study_amd import _native
from aws_training_study_amd.pcp_attention import (
    KVCacheWriter,
    PageAllocator,
    PCPAttentionConfig,
    append_history,
    build_page_pool,
    make_history_attention_kernel,
)
from aws_training_study_amd.pcp_attention.current import CurrentAttentionKernel

pytestmark = pytest.mark.gpu


def _case(device, kv_dtype="fp8_e4m3fn"):
    cfg = PCPAttentionConfig(pcp_size=2, current_len=128, max_history_len=512, actual_history_len=512, block_size=128,
                             interleave_size=64, num_q_heads=4, num_kv_heads=2, head_dim=64, backend="hip",
                             kv_dtype=kv_dtype).validate()
    gen = torch.Generator(device=device).manual_seed(1)

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=device, dtype=torch.bfloat16)

    table = torch.arange(cfg.num_pages, device=device, dtype=torch.int32).flip(0).reshape(2, -1).contiguous()
    pool, k_scale, v_scale, valid = build_page_pool(cfg, normal(2, 500, 64), normal(2, 500, 64), table)
    return cfg, normal(2, 4, 64, 64), pool, table, valid, k_scale, v_scale


@pytest.mark.parametrize("kv_dtype,precision,splits", [("fp8_e4m3fn", "auto", "auto"), ("fp8_e4m3fn", "fp8", 1),
                                                       ("fp8_e4m3fn", "bf16", 3), ("bfloat16", "auto", "auto")])
def test_history_common_form_equals_the_general_path(kv_dtype, precision, splits, cuda_device):
    cfg, q, pool, table, valid, k_scale, v_scale = _case(cuda_device, kv_dtype)
    kernel = make_history_attention_kernel(cfg)
    kw = dict(page_valid_len=valid, k_scale=k_scale, v_scale=v_scale, precision=precision, splits=splits)
    # an int64 copy of the lengths: the general path
    first = kernel(q, pool, table, return_lse=True, **dict(kw, page_valid_len=valid.long()))
    other = torch.empty_like(q)
    for _ in range(2):
        out, lse = kernel(q, pool, table, return_lse=True, **kw)
        assert torch.equal(out, first[0]) and torch.equal(lse, first[1])
        assert kernel(q, pool, table, out=other, **kw) is not None and torch.equal(other, first[0])
        assert torch.equal(kernel(q, pool, table.long(), **kw), first[0])
    # another stream gets a workspace of its own
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = kernel(q, pool, table, **kw)
    side.synchronize()
    assert torch.equal(out, first[0])
    # forms left to the general path
    assert torch.equal(kernel(q, pool, table.cpu(), **kw), first[0])
    kw_cpu = dict(kw, page_valid_len=valid.cpu().long(), k_scale=torch.tensor(k_scale), splits=splits)
    assert (kernel(q, pool, table, **kw_cpu).float() - first[0].float()).abs().max() <= 1e-2
    with pytest.raises(ValueError, match="q must be contiguous bfloat16"):
        kernel(q.transpose(2, 3), pool, table, **kw)
    with pytest.raises(ValueError, match="q must be contiguous bfloat16"):
        kernel(q.float(), pool, table, **kw)
    with pytest.raises(ValueError, match="GPU tensor"):
        kernel(q.cpu(), pool, table, **kw)
    with pytest.raises(ValueError, match="block_table must be"):
        kernel(q, pool, table[:, :-1].contiguous(), **kw)
    with pytest.raises(ValueError, match="kv_pages must be contiguous"):
        kernel(q, pool.view(torch.uint8), table, **kw)
    with pytest.raises(ValueError, match="out must be contiguous"):
        kernel(q, pool, table, out=other.float(), **kw)
    with pytest.raises(ValueError, match="not both"):
        kernel(q, pool, table, torch.zeros(2, 1, 1, 128), **kw)


def test_current_and_cache_calls(cuda_device):
    cfg, q, _, _, _, _, _ = _case(cuda_device)
    kv = torch.randn((2, 2, 128, 64), device=cuda_device, dtype=torch.bfloat16)
    step = CurrentAttentionKernel(cfg)
    out, lse = step(q, kv, return_lse=True)
    assert torch.equal(step(q, kv), out)
    with pytest.raises(ValueError, match="kv_current must be"):
        step(q, kv[:, :, :64].contiguous())
    with pytest.raises(ValueError, match="pass both"):
        step(q, kv, out)

    def fresh():
        allocator = PageAllocator(cfg, cuda_device)
        return (allocator, torch.zeros((cfg.num_pages, cfg.page_elements), dtype=torch.float8_e4m3fn,
                                       device=cuda_device), allocator.empty_table(),
                torch.zeros((2, cfg.max_local_blocks), dtype=torch.int32, device=cuda_device))

    x = torch.randn((2, 300, 64), device=cuda_device, dtype=torch.bfloat16)
    writer = KVCacheWriter(cfg)
    a, b = fresh(), fresh()
    append_history(writer, a[0], x, x, a[1], a[2], a[3], first_pos=7, k_scale=0.01, v_scale=0.02)
    # scales that are not Python floats: the general path
    append_history(writer, b[0], x, x, b[1], b[2], b[3], first_pos=7, k_scale=torch.tensor(0.01),
                   v_scale=torch.tensor(0.02))
    for s, t in zip(a[1:], b[1:]):
        assert torch.equal(s.view(torch.uint8), t.view(torch.uint8))
    assert int(a[0].free_count) == int(b[0].free_count) < cfg.num_pages
    with pytest.raises(ValueError, match="v must be a contiguous bfloat16"):
        writer(x, x[:, :5].contiguous(), a[1], a[2])
    with pytest.raises(ValueError, match="kv_pages must be"):
        writer(x, x, a[1].view(torch.uint8), a[2])
    with pytest.raises(RuntimeError, match="BAD_SHAPE"):
        writer(x, x, a[1], a[2], first_pos=400)
    with pytest.raises(RuntimeError, match="BAD_SHAPE"):
        a[0].allocate(400, 300, a[2])


# Pointer-sized arguments of the C entries behind the native calls.
C_ENTRY_ARGS = {"pcpa_history_attention_lse": 8, "pcpa_history_attention_split": 11, "pcpa_current_attention": 9,
                "pcpa_kv_cache_write": 10, "pcpa_page_alloc": 8}


@pytest.mark.parametrize("entry", sorted(C_ENTRY_ARGS))
def test_a_failed_launch_is_raised_and_not_made_again(entry, cuda_device, monkeypatch):
    """A status of the C entry is the call's error: kernels of it may be
    queued, so that the general path must not make the call a second time."""
    cfg, q, pool, table, valid, k_scale, v_scale = _case(cuda_device)
    calls = []

    def fail(*args):
        calls.append(entry)
        return next(code for code, name in _native.STATUS_NAMES.items() if name == "PCPA_ERR_LAUNCH")

    c_fail = ctypes.CFUNCTYPE(ctypes.c_int32, *[ctypes.c_void_p] * C_ENTRY_ARGS[entry])(fail)
    monkeypatch.setattr(_native, "function_address", lambda fn: ctypes.cast(c_fail, ctypes.c_void_p).value)
    x = torch.randn((2, 300, 64), device=cuda_device, dtype=torch.bfloat16)
    zeros = torch.zeros_like(table)
    with pytest.raises(_native.PcpaError, match="LAUNCH"):
        if entry.startswith("pcpa_history"):
            splits = 1 if entry.endswith("lse") else 2
            make_history_attention_kernel(cfg)(q, pool, table, page_valid_len=valid, k_scale=k_scale,
                                               v_scale=v_scale, precision="fp8", splits=splits)
        elif entry == "pcpa_current_attention":
            CurrentAttentionKernel(cfg)(q, x[None, :, :128].expand(2, -1, -1, -1).contiguous())
        elif entry == "pcpa_kv_cache_write":
            KVCacheWriter(cfg)(x, x, pool, table, page_valid_len=zeros)
        else:
            PageAllocator(cfg, cuda_device).allocate(0, 300, zeros - 1)
    assert calls == [entry]
    torch.cuda.synchronize()
    assert int(zeros.sum()) == 0


@pytest.mark.parametrize("kv_dtype,precision,splits", [("fp8_e4m3fn", "auto", "auto"), ("fp8_e4m3fn", "fp8", 1),
                                                       ("fp8_e4m3fn", "bf16", 3), ("bfloat16", "auto", "auto")])
def test_history_call_takes_the_common_form_only(kv_dtype, precision, splits, cuda_device):
    """The native call itself: it handles the common form (the general path
    would hide that it does not) and gives up every other one."""
    cfg, q, pool, table, valid, k_scale, v_scale = _case(cuda_device, kv_dtype)
    kernel = make_history_attention_kernel(cfg)
    want = kernel(q, pool, table, page_valid_len=valid.long(), k_scale=k_scale, v_scale=v_scale, precision=precision,
                  splits=splits)
    kernel(q, pool, table, page_valid_len=valid, k_scale=k_scale, v_scale=v_scale, precision=precision, splits=splits)
    call = kernel._plans[precision, "fast", splits]
    common = [q, pool, table, valid, k_scale, v_scale, None, False]

    def run(**changed):
        return call(*[changed.get(name, x) for name, x in zip(
            ("q", "pool", "table", "valid", "k_scale", "v_scale", "out", "lse"), common)])

    buffer = torch.empty_like(q)
    for kw in ({}, {"table": table.long()}, {"out": buffer}, {"q": q.clone().requires_grad_()},
               {"q": torch.nn.Parameter(q)}):
        out = run(**kw)
        assert type(out) is torch.Tensor and not out.requires_grad and torch.equal(out, want), kw
    assert run(out=buffer) is buffer
    out, lse = run(lse=True)
    assert torch.equal(out, want) and lse.shape == q.shape[:3] and lse.dtype == torch.float32

    class Subclass(torch.Tensor):
        pass

    for kw in ({"q": q.float()}, {"q": q.cpu()}, {"q": q.transpose(2, 3)}, {"q": q[:1]}, {"q": [q]},
               {"q": q.as_subclass(Subclass)}, {"pool": pool.view(torch.uint8)}, {"pool": pool[:, :-1]},
               {"table": table.cpu()}, {"table": table.float()}, {"table": table[:, :-1]}, {"valid": valid.long()},
               {"valid": valid.cpu()}, {"k_scale": 1}, {"v_scale": torch.tensor(v_scale)}, {"out": q.float()},
               {"out": q.cpu()}, {"lse": 1}):
        assert run(**kw) is None, kw
    seen = []
    torch.vmap(lambda x: (seen.append(run(q=x)), x)[1])(q[None])  # a batched tensor has no storage
    assert seen == [None]


def test_other_calls_take_the_common_form_only(cuda_device):
    cfg, q, pool, table, valid, _, _ = _case(cuda_device)
    kv = torch.randn((2, 2, 128, 64), device=cuda_device, dtype=torch.bfloat16)
    step = CurrentAttentionKernel(cfg)
    out, lse = step(q, kv, return_lse=True)
    assert torch.equal(step._fast(q, kv, None, None, None, False), out)
    merged, _ = step._fast(q, kv, out, lse, out.clone(), True)
    assert torch.equal(merged, step(q, kv, out, lse))
    for args in ((q.float(), kv, None, None, None, False), (q, kv[:1], None, None, None, False),
                 (q, kv, out, None, None, False), (q, kv, out, lse.double(), None, False),
                 (q, kv, None, None, out.cpu(), False), (q, kv, None, None, None, 1)):
        assert step._fast(*args) is None

    x = torch.randn((2, 300, 64), device=cuda_device, dtype=torch.bfloat16)
    writer = KVCacheWriter(cfg)
    writer(x, x, pool, table, page_valid_len=valid)
    common = (x, x, pool, table, 0, 1.0, 1.0, valid)
    assert writer._fast(*common) == 0 and writer._fast(*common[:-1], None) == 0
    assert writer._fast(x, x, pool, table.long(), *common[4:]) == 0
    for at, other in ((0, x.float()), (0, x[0]), (1, x[:, :5].contiguous()), (2, pool.view(torch.uint8)),
                      (3, table.cpu()), (4, -1), (4, 0.0), (4, 2**63), (5, 1), (6, torch.tensor(1.0)),
                      (7, valid.long())):
        assert writer._fast(*common[:at], other, *common[at + 1:]) is None, (at, other)

    allocator = PageAllocator(cfg, cuda_device)
    fresh = allocator.empty_table()
    allocator.allocate(0, 10, fresh)
    assert allocator._fast(0, 10, fresh, allocator.free_pages, allocator.free_count) == 0
    assert allocator._fast(0, 10, fresh.long(), allocator.free_pages, allocator.free_count) == 0
    for args in ((0, -1, fresh), (0.0, 10, fresh), (0, 2**31, fresh), (0, 10, fresh.cpu()), (0, 10, fresh[:, :1])):
        assert allocator._fast(*args, allocator.free_pages, allocator.free_count) is None, args


def test_threads_share_a_kernel_object(cuda_device):
    """Calls of several threads on streams of their own, native and general,
    with workspaces made and dropped meanwhile."""
    cfg, q, pool, table, valid, k_scale, v_scale = _case(cuda_device)
    kernel = make_history_attention_kernel(cfg)
    options = [dict(precision=p, splits=s) for p in ("auto", "fp8", "bf16") for s in (1, 2, 3)]
    kw = dict(k_scale=k_scale, v_scale=v_scale)
    want = [make_history_attention_kernel(cfg)(q, pool, table, page_valid_len=valid.long(), **kw, **o) for o in options]
    torch.cuda.synchronize()
    errors = []

    def work(offset):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                got = []
                for i in range(6 * len(options)):
                    o = (offset + i) % len(options)
                    lens = valid.long() if (offset + i) % 4 == 3 else valid
                    got.append((o, kernel(q, pool, table, page_valid_len=lens, **kw, **options[o])))
                torch.cuda.current_stream().synchronize()
                assert all(torch.equal(out, want[o]) for o, out in got)
        except BaseException as error:  # (raised in the test's own thread below)
            errors.append(error)

    threads = [threading.Thread(target=work, args=(3 * t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_an_interrupt_while_a_workspace_is_made_is_raised(cuda_device, monkeypatch):
    """Errors of the workspace's maker leave the call to the general path, an
    interrupt does not: it comes once."""
    cfg, q, pool, table, valid, k_scale, v_scale = _case(cuda_device)
    kernel = make_history_attention_kernel(cfg)
    kw = dict(page_valid_len=valid, k_scale=k_scale, v_scale=v_scale)
    make, raised = kernel._workspace, []

    def once(*args, error):
        if not raised:
            raised.append(error)
            raise error
        return make(*args)

    monkeypatch.setattr(kernel, "_workspace", lambda *args: once(*args, error=KeyboardInterrupt()))
    with pytest.raises(KeyboardInterrupt):
        kernel(q, pool, table, **kw)
    raised.clear()
    monkeypatch.setattr(kernel, "_workspace", lambda *args: once(*args, error=RuntimeError()))
    assert kernel(q, pool, table, **kw).shape == q.shape and raised
