"""Key-split prefill launches on the device (csrc/prefill_split.hpp): short chunks over
longer caches, whose rows are packed (token, query head) and whose keys are cut into
pieces merged by a combine kernel.  16-bit caches against the oracle at the f16 / bf16
bar of test_gpu_prefill.py, Q8 caches at 1e-5 against the oracle's attention over the rows
the device wrote: both bounds are those of the unsplit kernels, whose arithmetic a piece
keeps; the merge adds two f32 roundings per piece.
"""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_prefill import _assert_close, _case, _image_block_case  # noqa: E402

pytestmark = pytest.mark.gpu


# One token (a single partly filled 32-row group), group sizes 1, 3, 7, 8 and 16, KV head
# counts on each XCD mapping (16, 4, 1, 3), a last piece of one key, windows that start
# inside a tile and leave whole pieces unseen, more than four pieces (both combines).
@pytest.mark.parametrize("h,g,d,fmt_name,m,hist,window", [
    (32, 8, 128, "F16", 1, 1023, 0), (32, 8, 128, "F16", 64, 1985, 0), (16, 16, 128, "F16", 33, 1500, 0),
    (16, 1, 128, "BF16", 17, 1200, 0), (12, 4, 128, "F16", 100, 1437, 700), (9, 3, 128, "BF16", 130, 900, 0),
    (14, 2, 64, "F16", 203, 1800, 0), (14, 2, 64, "BF16", 5, 2044, 1111), (8, 4, 256, "F16", 129, 1000, 0),
    (8, 4, 256, "BF16", 77, 1100, 1024), (8, 1, 256, "F16", 2, 640, 0)])
def test_split_prefill_chunk(orc, dev, h, g, d, fmt_name, m, hist, window):
    from gguf_runner_amd import ffi
    fmt = getattr(orc, fmt_name)
    rows = sorted({hist, hist + m - 1, hist + m // 2, hist + m // 3})
    got, ref, _, vc = _case(orc, dev, m=hist + m, n_heads=h, n_kv=g, d=d, fmt=fmt, seed=m + hist,
                             rope_mode=ffi.ROPE_NEOX, theta=1e6, norm=d != 64, window=window,
                             base_chunks=[hist, m], attend_rows=np.asarray(rows))
    _assert_close(got[rows], ref[rows])
    assert np.array_equal(*vc)  # (the K rows are the prep pass's, which a split does not change)


@pytest.mark.parametrize("d,fmt_name,window", [(64, "F16", 0), (128, "F16", 300), (256, "BF16", 0)])
def test_split_prefill_image_block(orc, dev, d, fmt_name, window):
    from gguf_runner_amd import ffi
    got, ref = _image_block_case(orc, dev, hist=900, blk=70, n_heads=8, n_kv=2, d=d, fmt=getattr(orc, fmt_name),
                                 seed=d, window=window, rope_mode=ffi.ROPE_NEOX, theta=1e4)
    _assert_close(got, ref)


def test_split_prefill_gate_and_smaller_chunks_share_a_workspace(dev):
    """The output gate is applied once, by the combine (the gated output over sigmoid(gate)
    is the ungated one: f32 rounding of the same values), and a call made with the
    workspace of a longer chunk gives the same output."""
    from gguf_runner_amd import ffi, ops
    g = torch.Generator(device=dev).manual_seed(5)
    h, kv, d, m, hist = 16, 2, 128, 48, 1600
    rnd = lambda *s: torch.randn(s, generator=g, device=dev)
    q, k, v = rnd(m, h, d).half(), rnd(m, kv, d).half(), rnd(m, kv, d).half()
    kc, vc = rnd(hist + m, kv, d).half(), rnd(hist + m, kv, d).half()
    gate = rnd(m, h, d)
    outs = []
    for gt in (None, gate):
        out = torch.empty((m, h, d), device=dev)
        ops.PrefillCall(q, k, v, kc, vc, out, base_pos=hist, rope_mode=ffi.ROPE_NONE, out_gate=gt,
                        out_gate_row_stride=h * d, out_gate_head_stride=d)()
        outs.append(out)
    torch.testing.assert_close(outs[1], outs[0] * torch.sigmoid(gate), rtol=1e-5, atol=1e-6)
    big = [rnd(4096, n, d).half() for n in (h, kv, kv)]
    bc = [torch.zeros((4096, kv, d), dtype=torch.half, device=dev) for _ in range(2)]
    long_call = ops.PrefillCall(*big, *bc, torch.empty((4096, h, d), device=dev), rope_mode=ffi.ROPE_NONE)
    out = torch.empty((m, h, d), device=dev)
    call = ops.PrefillCall(q, k, v, kc, vc, out, base_pos=hist, rope_mode=ffi.ROPE_NONE)
    assert call.ws.numel() <= long_call.ws.numel()
    call.args.workspace = long_call.args.workspace
    call()
    torch.cuda.synchronize()
    assert torch.equal(out, outs[0])


@pytest.mark.parametrize("kv_dtype", ["F16", "BF16"])
def test_run_state_chunk_reserves_its_own_partials(dev, kv_dtype):
    """A run state's short first chunk, which is not cut along its keys, takes device memory
    for its rows (a few hundred KB), not for the partials that a cut one may have (69 MB at
    head_dim 128).  Bound: 8 MB, the allocator's granularity and the mapped buffer's."""
    from gguf_runner_amd import ffi, runtime as rt
    p = rt.Config(n_layers=1, n_heads=32, n_kv_heads=8, head_dim=128, seq_len=64,
                  kv_dtype=getattr(ffi, "DTYPE_" + kv_dtype), rope_mode=ffi.ROPE_NONE)
    rows = [np.ones((16, w), np.float32) for w in (p.q_dim, p.kv_dim, p.kv_dim)]
    rt.prefill_attention_chunk(p, rt.malloc_run_state(p), 0, 0, *rows)  # kernels loaded
    s = rt.malloc_run_state(p)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    rt.prefill_attention_chunk(p, s, 0, 0, *rows)
    assert free - torch.cuda.mem_get_info()[0] <= 8 << 20


@pytest.mark.parametrize("block,h,g,d,m,hist,window,image", [
    (False, 32, 8, 128, 64, 900, None, False), (True, 16, 16, 128, 3, 1000, None, False),
    (False, 14, 2, 64, 50, 1100, 777, False), (True, 8, 4, 256, 40, 600, None, False),
    (False, 8, 1, 256, 1, 700, None, True), (False, 9, 3, 128, 70, 800, 500, True)])
def test_split_q8_chunk(orc, dev, block, h, g, d, m, hist, window, image):
    from gguf_runner_amd import ffi, runtime as rt
    n = hist + m
    p = rt.Config(n_layers=1, n_heads=h, n_kv_heads=g, head_dim=d, seq_len=n, kv_dtype=ffi.DTYPE_Q8,
                  q8_block_scales=block, rope_mode=ffi.ROPE_NONE, layer_windows=[window])
    s = rt.malloc_run_state(p)
    rng = np.random.default_rng(hist + d)
    q, k, v = (rng.standard_normal((n, w)).astype(np.float32) for w in (p.q_dim, p.kv_dim, p.kv_dim))
    rt.prefill_attention_chunk(p, s, 0, 0, q[:hist], k[:hist], v[:hist])
    call = rt.prefill_image_block if image else rt.prefill_attention_chunk
    got = call(p, s, 0, hist, q[hist:], k[hist:], v[hist:])
    kq, vq = rt.read_kv_rows(p, s, 0, 0, n)
    ks, vs = rt.read_kv_scales(p, s, 0, 0, n)
    for i in sorted({0, m // 2, m - 1}):
        pos = hist + i
        start, end = (max(0, pos + 1 - window) if window else 0), pos + 1
        if image:
            start, end = min(start, hist), n
        ref = orc.attention_token(q[pos], kq, vq, orc.Q8B if block else orc.Q8, h, g, d, start, end,
                                  key_scale=ks.reshape(-1), value_scale=vs.reshape(-1))
        assert float(np.abs(got[i] - ref).max()) <= 1e-5, i
