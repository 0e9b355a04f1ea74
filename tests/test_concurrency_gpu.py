"""GPU test of concurrent calls from several host threads, each on its own stream.

The library keeps per-process state that concurrent callers share: the table
of side streams (one per caller stream, made on first use under a mutex) that
the seven-GEMM backward forks its dQ kernel onto, and the thread-local error
text and last split plans; every call takes its scratch from the caller's
workspace.  Eight jobs run at once, on as many host threads and streams, three
times each:
* a D = 64 backward that forks (``pick`` says so: no mask, 512 dK/dV
  workgroups of about 230 us), beside a causal one of that size that does not;
* a D = 128 five-GEMM backward (its dS tiles in the call's own workspace);
* a D = 96 backward and an fp32 one whose gradients are summed in chunks;
* a forward whose keys are split;
* a per-row-length decode;
* a paged decode.

Every result must equal, bit for bit, that of the same job run alone first:
each kernel's result is fixed by its inputs (no atomics, fixed split plans),
so any difference means two calls shared a buffer or an ordering they must
not.
"""

import threading

import pytest
import torch

from stackkernels_amd._core.attention.flash_bwd import flash_attn_bwd
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd
from stackkernels_amd._opt.pick import pick
from stackkernels_amd.torch import flash_decode

from _gpu_util import native_loaded

pytestmark = pytest.mark.gpu
ROUNDS = 3


def _rand(shape, dtype, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _train_job(b, hq, hkv, s, d, dtype, causal, seed):
    q, k, v, do = (_rand((b, h, s, d), dtype, seed + i)
                   for i, h in enumerate((hq, hkv, hkv, hq)))

    def run():
        # the launchers, not autograd: autograd would run every thread's
        # backward on its one device thread
        out, lse = flash_attn_fwd(q, k, v, is_causal=causal)
        return (out, lse, *flash_attn_bwd(do, q, k, v, out, lse, is_causal=causal))

    return run


def _split_job(seed):
    q, k, v = (_rand((1, h, s, 128), torch.bfloat16, seed + i)
               for i, (h, s) in enumerate(((32, 512), (8, 16000), (8, 16000))))
    return lambda: flash_attn_fwd(q, k, v, is_causal=True)


def _decode_job(paged, seed):
    dtype = torch.float16 if paged else torch.bfloat16
    b, hq, hkv, d = 8, 32, 8, 128
    q = _rand((b, hq, 1, d), dtype, seed)
    lens = torch.randint(0, 4096, (b,), generator=torch.Generator().manual_seed(seed)).int().cuda()
    if not paged:
        k, v = _rand((b, hkv, 4096, d), dtype, seed + 1), _rand((b, hkv, 4096, d), dtype, seed + 2)
        return lambda: (flash_decode(q, k, v, cache_seqlens=lens),)
    ps, per_row = 64, 64
    kp = _rand((b * per_row, hkv, ps, d), dtype, seed + 1)
    vp = _rand((b * per_row, hkv, ps, d), dtype, seed + 2)
    table = torch.randperm(b * per_row, generator=torch.Generator().manual_seed(seed))
    table = table.view(b, per_row).int().cuda()
    return lambda: (flash_decode(q, kp, vp, cache_seqlens=lens, block_table=table),)


def test_concurrent_threads_and_streams_match_serial_results(device):
    jobs = {
        "bwd_d64_forked": _train_job(2, 16, 8, 4096, 64, torch.bfloat16, False, 10),
        "bwd_d64_heavy_first": _train_job(2, 8, 8, 4096, 64, torch.bfloat16, True, 15),
        "bwd_d96_chunks": _train_job(1, 32, 8, 2000, 96, torch.bfloat16, True, 50),
        "bwd_f32_chunks": _train_job(2, 8, 8, 1024, 64, torch.float32, False, 60),
        "fwd_key_splits": _split_job(70),
        "bwd_d128_five_gemm": _train_job(1, 8, 2, 1024, 128, torch.float16, False, 20),
        "decode_varlen": _decode_job(False, 30),
        "decode_paged": _decode_job(True, 40),
    }
    def plan(op, b, h, s, d, **kw):
        return pick(op, (b, h, s, d), dtype=kw.pop("dtype", "bfloat16"), **kw)

    assert plan("flash_bwd", 2, 16, 4096, 64, num_kv_heads=8)["dq"]["side_stream"]
    assert plan("flash_bwd", 1, 32, 2000, 96, num_kv_heads=8, is_causal=True)["splits"] > 1
    assert plan("flash_bwd", 2, 8, 1024, 64, dtype="float32")["dq"]["splits"] > 1
    assert plan("flash_attn", 1, 32, 512, 128, num_kv_heads=8, kv_len=16000,
                is_causal=True)["SPLIT_KV"] > 1
    expect = {name: job() for name, job in jobs.items()}
    torch.cuda.synchronize()
    assert native_loaded()

    got = {name: [] for name in jobs}
    errors = []
    start = threading.Barrier(len(jobs))

    def worker(name):
        try:
            stream = torch.cuda.Stream()
            start.wait()
            with torch.cuda.stream(stream):
                for _ in range(ROUNDS):
                    got[name].append(jobs[name]())
            stream.synchronize()
        except Exception as e:  # noqa: BLE001 -- reported by the main thread
            errors.append(f"{name}: {e!r}")

    threads = [threading.Thread(target=worker, args=(n,)) for n in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=120)
    assert not any(t.is_alive() for t in threads), "a worker thread did not finish"
    torch.cuda.synchronize()
    assert not errors, errors
    for name, runs in got.items():
        assert len(runs) == ROUNDS, name
        for r, outs in enumerate(runs):
            for i, (a, b) in enumerate(zip(outs, expect[name])):
                assert torch.equal(a, b), f"{name}, round {r}, output {i} differs from the serial run"
