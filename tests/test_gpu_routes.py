"""GPU: which kernels a call launches, where the choice between two of them rests on which
is faster for its sizes.  The names come from torch's profiler, which sees every launch of
the process."""
import pytest

import oracle as O
import puter_amd

pytestmark = pytest.mark.gpu


def launched(call):
    """The names of the kernels that call launches."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    return [e.name for e in p.events() if "puter::" in e.name or "_kernel" in e.name]


def grids(call):
    """The blocks of the kernels that call launches."""
    import json
    import os
    import tempfile
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "trace.json")
        p.export_chrome_trace(path)
        with open(path) as f:
            events = json.load(f)["traceEvents"]
    found = [e["args"]["grid"] for e in events if e.get("cat") == "kernel" and "puter::" in e["name"]]
    return [x * y * z for x, y, z in found]


def zeros(dt, *shape):
    import torch
    t = {O.F32: torch.float32, O.BF16: torch.bfloat16, O.F16: torch.float16}[dt]
    return torch.zeros(shape, dtype=t, device="cuda")


@pytest.mark.parametrize("op,dt,rows,h,kernel", [
    # short rows: a wave each, four to a block
    ("rms", O.F32, 4096, 512, "norm_wave"), ("ln", O.F32, 1, 512, "norm_wave"), ("rms", O.BF16, 16, 1024, "norm_wave"),
    ("gr_ln", O.F32, 16, 512, "norm_wave"), ("adaptive", O.F32, 16, 512, "norm_line"),
    # tensors past the L2s
    ("ln", O.F32, 2048, 4096, "norm_wave"), ("rms", O.BF16, 2048, 8192, "norm_wave"),
    ("rms", O.BF16, 3500, 4096, "norm_wave"), ("adaptive", O.BF16, 6000, 2048, "norm_wave"),
    # few rows, other lengths, and f16
    ("rms", O.BF16, 1, 4096, "norm_line"), ("ln", O.BF16, 1024, 8192, "norm_line"),
    ("ln", O.BF16, 4096, 3072, "norm_line"), ("rms", O.F16, 2048, 8192, "norm_line"),
    ("gr_rms", O.F16, 16, 1024, "norm_line"), ("gr_rms", O.F16, 1024, 2048, "norm_wave"),
    ("rms", O.BF16, 16384, 4096, "norm_row"),
])
def test_norm_kernels(backend, op, dt, rows, h, kernel):
    x, y, z, g, mod = zeros(dt, rows, h), zeros(dt, rows, h), zeros(dt, rows, h), zeros(dt, h), zeros(dt, 1, 3 * h)
    cfg = puter_amd.RMSNormConfig(1e-5)
    names = launched({
        "rms": lambda: backend.RMSNorm(cfg, x, g, y, rows, h, dt),
        "ln": lambda: backend.LayerNorm(x, g, g, y, rows, h, dt),
        "adaptive": lambda: backend.AdaptiveRMSNorm(cfg, x, mod, y, rows, h, rows, 3 * h, dt),
        "gr_rms": lambda: backend.GatedResidualRMSNorm(cfg, x, x, mod, g, y, z, rows, h, rows, 3 * h, 0, dt),
        "gr_ln": lambda: backend.GatedResidualLayerNorm(x, x, mod, g, g, y, z, rows, h, rows, 3 * h, 0, dt),
    }[op])
    names = [n for n in names if "puter::" in n]
    assert len(names) == 1 and kernel in names[0], names


@pytest.mark.parametrize("dt,rows,inner,cols,kernels", [
    (O.BF16, 1, 4096, 4096, ["matmul_rows"]), (O.BF16, 32, 4096, 4096, ["matmul_rows"]),
    # one slice of K, or a round of column tiles: the skinny kernel unsplit
    (O.BF16, 32, 64, 1024, ["matmul_skinny"]), (O.F16, 4, 32, 4096, ["matmul_skinny"]),
    (O.BF16, 32, 1024, 65536, ["matmul_skinny"]), (O.BF16, 8, 4096, 33000, ["matmul_skinny"]),
    (O.BF16, 8, 4096, 80000, ["matmul_rows"]), (O.BF16, 8, 64, 131072, ["matmul_rows"]),
    (O.BF16, 64, 4096, 4096, ["matmul_skinny", "matmul_splitk_reduce"]),
    # unaligned: the generic kernel where K is small
    (O.BF16, 65, 5, 33, ["matmul_generic"]), (O.BF16, 20, 15, 129, ["matmul_generic"]),
    (O.F16, 4, 5, 33, ["matmul_generic"]), (O.BF16, 200, 31, 129, ["matmul_generic"]),
    (O.BF16, 7, 31, 33, ["matmul_rows"]), (O.F16, 200, 31, 129, ["matmul_rows"]),
    (O.BF16, 1000, 31, 4097, ["matmul_rows"]), (O.BF16, 33, 4096, 32001, ["matmul_rows"]),
    # 256 x 256 tiles with K in two halves, where they fill half a round or one and a half
    (O.BF16, 2041, 8200, 4088, ["64, 2, true>"]), (O.F16, 2817, 8192, 8192, ["64, 2, true>"]),
    (O.BF16, 4100, 7752, 4096, ["64, 2, true>"]), (O.BF16, 1793, 16384, 4096, ["matmul_skinny"]),
    (O.BF16, 4096, 4096, 4096, ["64, 2, false>"]),
])
def test_matmul_kernels(backend, dt, rows, inner, cols, kernels):
    a, b, c = zeros(dt, rows, inner), zeros(dt, inner, cols), zeros(dt, rows, cols)
    backend.Matmul(c, a, b, rows, inner, cols, dt)   # (the scratch is there)
    names = launched(lambda: backend.Matmul(c, a, b, rows, inner, cols, dt))
    assert len(names) == len(kernels) and all(k in n for k, n in zip(kernels, names)), names


@pytest.mark.parametrize("dt,seq_q,seq_k,dim,causal,kernel", [
    # rows that see a few keys: the general kernel
    (O.F32, 4, 1000, 64, True, "flash_generic"), (O.BF16, 1, 1000, 40, True, "flash_generic"),
    (O.BF16, 20, 1000, 512, True, "flash_generic"), (O.BF16, 1000, 1, 40, False, "flash_generic"),
    (O.F32, 24, 1000, 64, True, "flash_score"), (O.F32, 1, 1000, 64, False, "flash_score"),
    (O.BF16, 40, 1000, 512, True, "flash_score"), (O.BF16, 4, 1000, 40, True, "prefill_kernel"),
    (O.F16, 4, 1, 256, False, "prefill_kernel"),
])
def test_flash_kernels(backend, dt, seq_q, seq_k, dim, causal, kernel):
    q, k, out = zeros(dt, seq_q, dim), zeros(dt, seq_k, dim), zeros(dt, seq_q, dim)
    cfg = puter_amd.FlashAttentionConfig(64, causal)
    call = lambda: backend.FlashAttention(cfg, q, k, k, out, seq_q, seq_k, dim, dim, dt)  # noqa: E731
    call()   # (the scratch is there)
    names = launched(call)
    assert kernel in names[0], names


def mha(backend, dt, seq_q, seq_k, heads, dim, kv_heads=None):
    q, kv, out = zeros(dt, seq_q, heads * dim), zeros(dt, seq_k, (kv_heads or heads) * dim), zeros(dt, seq_q, heads * dim)
    cfg = puter_amd.MultiHeadAttentionConfig(heads, dim, True, 0, 0.0, kv_heads or heads)
    call = lambda: backend.MultiHeadAttention(cfg, q, kv, kv, out, seq_q, seq_k, dt)  # noqa: E731
    call()
    return launched(call)


def test_split_f32_attention_combines_by_head_dim(backend):
    """The sums of a split are folded by a kernel of the head dim's own, whose loads the
    compiler can issue ahead of each other."""
    names = mha(backend, O.F32, 16, 3000, 8, 128)
    assert len(names) == 2 and "prefill_f32_combine_kernel<128" in names[1], names


@pytest.mark.parametrize("dt,seq_q,seq_k,heads,dim,kernel", [
    # few rows of head dims other than 64 and 128: a block per row
    (O.BF16, 8, 200, 8, 256, "mha_"), (O.BF16, 2, 700, 8, 256, "mha_"), (O.BF16, 16, 200, 8, 40, "mha_"),
    (O.F32, 16, 700, 32, 256, "mha_"), (O.F32, 64, 200, 32, 160, "mha_"), (O.F32, 64, 512, 1, 16, "mha_"),
    # many, or over many keys
    (O.BF16, 300, 700, 8, 96, "prefill_kernel"), (O.BF16, 8, 3000, 8, 256, "prefill_kernel"),
    (O.BF16, 8, 40, 8, 40, "prefill_kernel"), (O.F16, 8, 200, 8, 256, "prefill_kernel"),
    (O.F32, 300, 700, 16, 96, "prefill_f32_kernel"), (O.F32, 16, 2000, 8, 40, "prefill_f32_kernel"),
    (O.F32, 16, 3000, 8, 128, "prefill_f32_kernel"),
])
def test_attention_kernels(backend, dt, seq_q, seq_k, heads, dim, kernel):
    names = mha(backend, dt, seq_q, seq_k, heads, dim)
    assert kernel in names[0], names


@pytest.mark.parametrize("rows,inner,blocks", [(3, 64, 1), (4, 1024, 1), (16, 64, 2), (8, 2048, 4), (64, 1024, 32),
                                               (1025, 64, 129)])
def test_page_write_blocks(backend, rows, inner, blocks):
    """A handful of small rows is written by one block, more rows by two to a block."""
    import torch
    pool, values = zeros(O.BF16, 128, 16, inner), zeros(O.BF16, rows, inner)
    at = torch.arange(rows, dtype=torch.int32, device="cuda")
    ids, slots = at // 16, at % 16
    call = lambda: backend.KVPageWrite(pool, values, ids, slots, pool, 128, 16, inner, rows, 0, O.BF16)  # noqa: E731
    assert grids(call) == [blocks]
