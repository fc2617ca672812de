"""The native argument checks (_tq4_host) against the Python ones: a valid call
gives the same bits either way, and a call that Python refuses is refused with
the same message (the native function then takes nothing)."""
import math
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _bytes(n):
    return torch.randint(-128, 128, (n,), dtype=torch.int8, device=DEV)


def _calls():
    """{entry: (args, kwargs)} of one valid call each, on fresh tensors."""
    torch.manual_seed(7)
    H, d, S, P, T, B, G, K = 2, 64, 16, 8, 32, 2, 3, 2
    rows = P * H * S
    cache = [_bytes(rows * d // 2), _bytes(rows * d // 2), torch.rand(2 * rows, device=DEV)]
    signs = (torch.randint(0, 2, (d,), device=DEV) * 2 - 1).float()
    slots = torch.arange(T, dtype=torch.int32, device=DEV)
    bf = lambda *s: torch.randn(s, device=DEV).to(torch.bfloat16)  # noqa: E731
    a8 = lambda: torch.randint(-127, 128, (T, H, d), dtype=torch.int8, device=DEV)  # noqa: E731
    q, bt = bf(B, H * G, d), torch.randperm(P, device=DEV).to(torch.int32).view(B, P // B)
    cl = torch.tensor([50, 7], dtype=torch.int32, device=DEV)
    rec = torch.randn((B, H * G, K, d + 4), device=DEV)
    tabs = torch.ones(32 * d, dtype=torch.int8, device=DEV)
    dec = (q, *cache, bt, cl, signs, H, S, P)
    nz_rows = P * 64
    nz = [torch.randint(0, 256, (nz_rows * H * 128,), dtype=torch.uint8, device=DEV),
          torch.randint(0, 256, (nz_rows * H * 128,), dtype=torch.uint8, device=DEV),
          torch.rand((nz_rows, 8), device=DEV) + 0.5, bt, cl]
    q4, s256 = torch.randn((B, H * G, 256), device=DEV), torch.ones(256, device=DEV)
    zero = lambda: torch.zeros(1 << 20, dtype=torch.uint8, device=DEV)  # noqa: E731
    rms = [_bytes(rows * d // 2), _bytes(rows * d // 2), torch.rand(P * S * 8, device=DEV)]
    return {
        "reshape_and_cache_a8": ((a8(), a8(), *cache, slots), dict(pi_signs=signs)),
        "reshape_and_cache_a8:tables": ((a8(), a8(), *cache, slots), dict(tables=tabs)),
        "reshape_and_cache_bf16": ((bf(T, H, d), bf(T, H, d), *cache, slots),
                                   dict(pi_signs=signs, num_blocks=P, block_size=S)),
        "reshape_scatter": ((bf(T, H, d), bf(T, H, d), *cache, slots, signs),
                            dict(cu_seqlens=torch.tensor([0, 16, T], dtype=torch.int32, device=DEV))),
        "reshape_scatter:tokens": ((bf(8, H, d), bf(8, H, d), *cache, slots[:8] * 16, signs),
                                   dict(num_blocks=P, inv_sqrt_len=0.125)),
        "paged_decode": (dec, dict(num_splits=K, workspace=zero())),
        "paged_decode:gate": (dec, dict(num_splits=1, output_stage=2, gate=torch.randn(
            q.shape, device=DEV), out=torch.empty_like(q))),
        "paged_decode_partials": (dec, dict(num_splits=K)),
        "splitk_combine": ((rec, signs, B, H * G, d, K), {}),
        "rms_reshape_and_cache": ((bf(T, H, d), bf(T, H, d), *rms, slots, signs), {}),
        "kv4fp8_decode": ((q4, *nz, H, 64, P), dict(workspace=zero())),
        "kv4fp8_decode_raw_query": ((q4.half(), s256, *nz, H, 64, P),
                                    dict(workspace=zero(), output_stage=1,
                                         query_out=torch.empty_like(q4))),
        "icdf_quantize": ((torch.randn(2048, device=DEV).half(),), {}),
        "lloydmax_quantize": ((torch.randn(64, device=DEV),), dict(bits=2)),
        "lloydmax_quantize:decode": ((torch.arange(16, dtype=torch.uint8, device=DEV),),
                                     dict(mode=4)),
    }


def _run(tq4, name, args, kwargs, native):
    mod = sys.modules[tq4.__name__ + ".tq4"]
    keep = mod._fast
    assert keep is not None, "_tq4_host.so is not built"
    if not native:
        mod._fast = None
    try:
        r = getattr(tq4, name.split(":")[0])(*args, **kwargs)
        torch.cuda.synchronize()
        outs = [x for x in (r if isinstance(r, tuple) else (r,)) if x is not None]
        return outs + [x for x in (*args, *kwargs.values()) if isinstance(x, torch.Tensor)]
    except Exception as e:  # noqa: BLE001
        return type(e).__name__, str(e)
    finally:
        mod._fast = keep


NAMES = ["reshape_and_cache_a8", "reshape_and_cache_a8:tables", "reshape_and_cache_bf16",
         "reshape_scatter", "reshape_scatter:tokens", "paged_decode", "paged_decode:gate",
         "paged_decode_partials", "splitk_combine", "rms_reshape_and_cache", "kv4fp8_decode",
         "kv4fp8_decode_raw_query", "icdf_quantize", "lloydmax_quantize",
         "lloydmax_quantize:decode"]


@pytest.mark.parametrize("name", NAMES)
def test_valid_call_same_bits(tq4, name):
    tq4.lib()
    got = [_run(tq4, name, *_calls()[name], native) for native in (True, False)]
    assert isinstance(got[0], list) and isinstance(got[1], list), got
    for a, b in zip(*got):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert np.array_equal(a.contiguous().view(torch.uint8).cpu().numpy(),
                              b.contiguous().view(torch.uint8).cpu().numpy())


def _bad(key, v):
    """What the checks refuse in place of a tensor argument."""
    yield v.cpu()
    yield v.to(torch.float64)
    if key != "workspace":  # half of this one is still enough
        yield v.reshape(-1)[:max(1, v.numel() // 2 - 1)].contiguous()
    if v.dim() > 1:
        yield v.transpose(0, v.dim() - 1)
    yield None
    yield "text"


@pytest.mark.parametrize("name", NAMES)
def test_refused_call_same_message(tq4, name):
    """Each tensor argument in turn on the host, of another dtype, short, not
    contiguous, None or no tensor at all: where Python refuses the call, the
    native route ends in the same refusal."""
    tq4.lib()
    args, kwargs = _calls()[name]
    refused = 0
    for key in (*range(len(args)), *kwargs):
        v = args[key] if isinstance(key, int) else kwargs[key]
        if not isinstance(v, torch.Tensor):
            continue
        for bad in _bad(key, v):
            a, k = list(args), dict(kwargs)
            if isinstance(key, int):
                a[key] = bad
            else:
                k[key] = bad
            want = _run(tq4, name, a, k, native=False)
            if isinstance(want, tuple):
                refused += 1
                assert _run(tq4, name, a, k, native=True) == want, (key, want)
    assert refused or name.startswith(("icdf", "lloyd"))


@pytest.mark.parametrize("name", NAMES)
def test_refused_number_same_message(tq4, name):
    """Each size argument, and the pool's page count and page size together, at
    zero and so large that the pool's size passes 2^64: where Python refuses the
    call, the native route ends in the same refusal."""
    import inspect
    tq4.lib()
    args, kwargs = _calls()[name]
    bound = inspect.signature(getattr(tq4, name.split(":")[0])).bind(*args, **kwargs)
    bound.apply_defaults()
    call = dict(bound.arguments)
    numbers = [k for k in ("num_blocks", "block_size", "num_kv_heads", "kv_heads", "num_requests",
                           "num_seqs", "num_heads", "head_size") if k in call]
    big = (1 << 30, (1 << 31) - 1, 1 << 31, 1 << 40)
    tries = [{k: v} for k in numbers for v in (0, *big)]
    if "num_blocks" in call:
        tries += [dict(num_blocks=a, block_size=b) for a in (1, *big) for b in big]
    refused = 0
    for over in tries:
        want = _run(tq4, name, (), {**call, **over}, native=False)
        if isinstance(want, tuple):
            refused += 1
            assert _run(tq4, name, (), {**call, **over}, native=True) == want, over
    assert refused or not numbers


def test_other_streams_and_threads(tq4):
    """The call goes to torch's current stream of its thread, or the one given."""
    import threading
    q = torch.randn((1, 4, 64), device=DEV).to(torch.bfloat16)
    rec = torch.randn((1, 4, 2, 68), device=DEV)
    signs = torch.ones(64, device=DEV)
    want = tq4.splitk_combine(rec, signs, 1, 4, 64, 2)
    got = []

    def work():
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            got.append(tq4.splitk_combine(rec, signs, 1, 4, 64, 2, out=torch.empty_like(q)))
        got.append(tq4.splitk_combine(rec, signs, 1, 4, 64, 2, stream=s))
        s.synchronize()

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert len(got) == 6 and all(torch.equal(g, want) for g in got)
    assert math.isfinite(float(want.float().sum()))


@pytest.mark.parametrize("name", ["paged_decode", "paged_decode_partials", "splitk_combine",
                                  "kv4fp8_decode", "icdf_quantize", "lloydmax_quantize"])
def test_exception_of_an_allocation(tq4, name):
    """An exception that Python code raises out of the output's allocation (here a
    dispatch mode) reaches the caller as it is."""
    from torch.utils._python_dispatch import TorchDispatchMode
    tq4.lib()

    class Refuse(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if "empty" in str(func):
                raise KeyError("no allocation here")
            return func(*args, **(kwargs or {}))

    args, kwargs = _calls()[name]
    torch.cuda.synchronize()
    with Refuse():
        got = [_run(tq4, name, args, kwargs, native) for native in (False, True)]
    assert got[0] == got[1] == ("KeyError", repr("no allocation here"))
