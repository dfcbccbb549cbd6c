"""Gated DeltaNet parity: gr_deltanet_attention (recurrent and chunk-64 HIP paths)
vs the CPU oracle's token-serial recurrence (qwen3next_state_head_step,
reference math.rs:492-546, per token as inference.rs:2866-2885).

Tolerance (fp32 state path, fixed before measuring): max |gpu - ref| <= 1e-5 for
outputs and final state."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _inputs(orc, T, H, d, seed, fmt):
    rng = np.random.default_rng(seed)
    conv = {orc.F32: lambda x: x, orc.F16: orc.f16_bits, orc.BF16: orc.bf16_bits}[fmt]
    q = conv(rng.standard_normal((T, H, d), dtype=np.float32))
    k = conv(rng.standard_normal((T, H, d), dtype=np.float32))
    v = conv(rng.standard_normal((T, H, d), dtype=np.float32))
    beta = (1.0 / (1.0 + np.exp(-rng.standard_normal((T, H))))).astype(np.float32)
    gate = rng.uniform(-0.1, 0.0, (T, H)).astype(np.float32)
    return q, k, v, gate, beta


def _to_dev(x, fmt, orc, dev):
    if fmt == orc.F32:
        return torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    dt = torch.float16 if fmt == orc.F16 else torch.bfloat16
    return torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).view(dt).to(dev)


def _run(orc, dev, T, H, d, seed, fmt, algo, state0=None, chunks=None):
    from gguf_runner_amd import ops
    q, k, v, gate, beta = _inputs(orc, T, H, d, seed, fmt)
    S0 = np.zeros((H, d, d), np.float32) if state0 is None else state0
    ref, Sref = orc.deltanet_scan(orc.upcast(q, fmt), orc.upcast(k, fmt), orc.upcast(v, fmt),
                                  gate, beta, S0, eps=1e-6, n_threads=orc.env_threads())
    st = torch.from_numpy(S0.copy()).to(dev)
    qd, kd, vd = (_to_dev(x, fmt, orc, dev) for x in (q, k, v))
    gd = torch.from_numpy(gate).to(dev)
    bd = torch.from_numpy(beta).to(dev)
    out = torch.empty((T, H, d), dtype=torch.float32, device=dev)
    b = 0
    for c in (chunks or [T]):
        o = torch.empty((c, H, d), dtype=torch.float32, device=dev)
        ops.DeltaNetCall(qd[b:b + c].contiguous(), kd[b:b + c].contiguous(),
                         vd[b:b + c].contiguous(), gd[b:b + c].contiguous(),
                         bd[b:b + c].contiguous(), st, o, algo=algo)()
        out[b:b + c] = o
        b += c
    torch.cuda.synchronize()
    return out.cpu().numpy(), ref, st.cpu().numpy(), Sref


@pytest.mark.parametrize("algo", [1, 2])
def test_config5_deltanet_prefill_4096(orc, dev, algo):
    """Config 5: 16 heads, d128, fp32 state, 4096-token prefill (chunk 64), bf16 inputs,
    q/k L2-normed in-kernel, beta = sigmoid(N(0,1)), log-decay ~U(-0.1, 0)."""
    got, ref, S, Sref = _run(orc, dev, 4096, 16, 128, 1005, orc.BF16, algo)
    assert float(np.abs(got - ref).max()) <= TOL, np.abs(got - ref).max()
    assert float(np.abs(S - Sref).max()) <= TOL, np.abs(S - Sref).max()


def test_config5_deltanet_decode_steps_after_prefill(orc, dev):
    """Config 5 as one sequence: the 4096-token chunked prefill, then 512 single-token
    recurrent decode steps on the state it leaves, against one token-serial scan
    over all 4608 tokens."""
    got, ref, S, Sref = _run(orc, dev, 4096 + 512, 16, 128, 1015, orc.BF16, 0,
                             chunks=[4096] + [1] * 512)
    assert float(np.abs(got - ref).max()) <= TOL, np.abs(got - ref).max()
    assert float(np.abs(S - Sref).max()) <= TOL, np.abs(S - Sref).max()


@pytest.mark.parametrize("T", [1, 5, 63, 64, 65, 200])
@pytest.mark.parametrize("algo", [1, 2])
def test_deltanet_ragged_lengths(orc, dev, T, algo):
    """Partial chunks (padded with beta = 0, gate = 0) and short sequences, f32 inputs,
    non-zero initial state."""
    rng = np.random.default_rng(T)
    S0 = (0.1 * rng.standard_normal((4, 128, 128))).astype(np.float32)
    got, ref, S, Sref = _run(orc, dev, T, 4, 128, 77 + T, orc.F32, algo, state0=S0)
    assert float(np.abs(got - ref).max()) <= TOL, np.abs(got - ref).max()
    assert float(np.abs(S - Sref).max()) <= TOL, np.abs(S - Sref).max()


def test_deltanet_nonfinite_inputs_follow_reference_guards(orc, dev):
    """Non-finite inputs take the reference's per-token guards (math.rs:523-545 and
    833-874: finite_or_zero on the normalised q / k, on v, on exp(gate), on beta, on
    kv, delta and o) on the chunked path too: the scan stops before a chunk with a
    non-finite value and the step kernel continues from its first token.  One event
    per head: NaN v element, inf k element, NaN q element, NaN gate, inf beta,
    gate +100 (exp overflows, g = 0 zeroes the state), one in the ragged last chunk."""
    T, H, d = 1000, 16, 128
    q, k, v, gate, beta = _inputs(orc, T, H, d, 4242, orc.F32)
    v[100, 3, 7] = np.nan
    k[300, 5, 11] = np.inf
    q[450, 7, 0] = np.nan
    gate[500, 9] = np.nan
    beta[700, 11] = np.inf
    gate[400, 1] = 100.0
    beta[990, 13] = np.nan
    S0 = (0.05 * np.random.default_rng(1).standard_normal((H, d, d))).astype(np.float32)
    ref, Sref = orc.deltanet_scan(q, k, v, gate, beta, S0, eps=1e-6, n_threads=orc.env_threads())
    assert np.isfinite(ref).all() and np.isfinite(Sref).all()
    from gguf_runner_amd import ops
    st = torch.from_numpy(S0.copy()).to(dev)
    out = torch.empty((T, H, d), dtype=torch.float32, device=dev)
    ops.DeltaNetCall(*(torch.from_numpy(x).to(dev) for x in (q, k, v, gate, beta)), st, out,
                     algo=2)()
    torch.cuda.synchronize()
    got, S = out.cpu().numpy(), st.cpu().numpy()
    assert np.isfinite(got).all() and np.isfinite(S).all()
    assert float(np.abs(got - ref).max()) <= TOL, np.abs(got - ref).max()
    assert float(np.abs(S - Sref).max()) <= TOL, np.abs(S - Sref).max()
    # the events matter: the state of head 1 restarts from zero at token 400
    assert float(np.abs(Sref[1]).max()) < float(np.abs(Sref[0]).max())


@pytest.mark.parametrize("fmt", ["F16", "BF16"])
@pytest.mark.parametrize("l2norm", [True, False])
def test_deltanet_16bit_inputs_chunked(orc, dev, fmt, l2norm):
    """16-bit q/k/v on the chunked path (exact 16-bit Gram products, raw-row MFMA
    operands), a ragged last chunk, non-zero initial state, with and without the
    fused normalisation (without it the oracle gets rows of norm ~1 so the
    recurrence stays in range)."""
    f = getattr(orc, fmt)
    T, H, d = 200, 4, 128
    q, k, v, gate, beta = _inputs(orc, T, H, d, 300 + int(l2norm), f)
    if not l2norm:  # unit-norm-ish rows stored in the 16-bit format
        conv = orc.f16_bits if f == orc.F16 else orc.bf16_bits
        rng = np.random.default_rng(9)
        qq = rng.standard_normal((T, H, d)).astype(np.float32)
        kk = rng.standard_normal((T, H, d)).astype(np.float32)
        q = conv(qq / np.linalg.norm(qq, axis=-1, keepdims=True) / np.sqrt(d))
        k = conv(kk / np.linalg.norm(kk, axis=-1, keepdims=True))
    S0 = (0.1 * np.random.default_rng(3).standard_normal((H, d, d))).astype(np.float32)
    ref, Sref = orc.deltanet_scan(orc.upcast(q, f), orc.upcast(k, f), orc.upcast(v, f), gate, beta, S0,
                                  l2norm=l2norm, eps=1e-6, n_threads=orc.env_threads())
    from gguf_runner_amd import ops
    st = torch.from_numpy(S0.copy()).to(dev)
    out = torch.empty((T, H, d), dtype=torch.float32, device=dev)
    ops.DeltaNetCall(_to_dev(q, f, orc, dev), _to_dev(k, f, orc, dev), _to_dev(v, f, orc, dev),
                     torch.from_numpy(gate).to(dev), torch.from_numpy(beta).to(dev), st, out,
                     l2norm=l2norm, algo=2)()
    torch.cuda.synchronize()
    got, S = out.cpu().numpy(), st.cpu().numpy()
    assert float(np.abs(got - ref).max()) <= TOL, np.abs(got - ref).max()
    assert float(np.abs(S - Sref).max()) <= TOL, np.abs(S - Sref).max()


@pytest.mark.parametrize("T", [1, 63, 64, 65, 128, 129, 321])
def test_deltanet_bf16_scan_chunk_edges(orc, dev, T):
    """The bf16 scan (state in registers, operands loaded a chunk ahead): one chunk, whole
    chunks, one row past a chunk, odd and even chunk counts; f32 arithmetic bar."""
    rng = np.random.default_rng(T)
    S0 = (0.1 * rng.standard_normal((3, 128, 128))).astype(np.float32)
    got, ref, S, Sref = _run(orc, dev, T, 3, 128, 40 + T, orc.BF16, 2, state0=S0)
    assert float(np.abs(got - ref).max()) <= TOL, np.abs(got - ref).max()
    assert float(np.abs(S - Sref).max()) <= TOL, np.abs(S - Sref).max()


def test_deltanet_bf16_scan_nonfinite(orc, dev):
    """Non-finite values in the bf16 scan: inputs (flagged by the prep, in the first, a
    middle and the ragged last chunk) and a state column that overflows inside the scan
    (gates above zero): its column block continues token by token from that chunk.
    Every other column keeps the f32 bar; of the overflowing one the outputs stay finite
    (where a sum overflows depends on its order) and the state ends infinite, as the
    reference's."""
    T, H, d = 500, 6, 128
    q, k, v, gate, beta = _inputs(orc, T, H, d, 99, orc.BF16)
    nan, inf = orc.bf16_bits(np.array([np.nan, np.inf], np.float32))
    v[3, 0, 7] = nan
    k[200, 1, 11] = inf
    q[499, 2, 0] = nan
    gate[260, 3] = np.nan
    S0 = (0.05 * np.random.default_rng(1).standard_normal((H, d, d))).astype(np.float32)
    gate[:300, 4] = 0.15
    gate[300, 4] = -90.0
    S0[4, :, 21] = 1e33
    ref, Sref = orc.deltanet_scan(*(orc.upcast(x, orc.BF16) for x in (q, k, v)), gate, beta, S0, eps=1e-6,
                                  n_threads=orc.env_threads())
    from gguf_runner_amd import ops
    st = torch.from_numpy(S0.copy()).to(dev)
    out = torch.empty((T, H, d), dtype=torch.float32, device=dev)
    ops.DeltaNetCall(*(_to_dev(x, orc.BF16, orc, dev) for x in (q, k, v)), torch.from_numpy(gate).to(dev),
                     torch.from_numpy(beta).to(dev), st, out, algo=2)()
    torch.cuda.synchronize()
    got, S = out.cpu().numpy(), st.cpu().numpy()
    assert np.isfinite(got).all()
    cols = np.ones((H, d), bool)
    cols[4, 21] = False
    # head 4's other columns grow with the gates too (to ~1e17): relative to their size
    tol = TOL * np.maximum(1.0, np.abs(np.where(cols, ref, 0)).max(axis=2, keepdims=True))
    assert (np.abs(got - ref) <= tol)[:, cols].all()
    S, Sref = S.transpose(0, 2, 1), Sref.transpose(0, 2, 1)  # [head][column][row]
    assert (np.abs(S[cols] - Sref[cols]) <= TOL * np.maximum(1.0, np.abs(Sref[cols]))).all()
    assert np.isinf(S[4, 21]).all() and np.isinf(Sref[4, 21]).all()


def test_deltanet_bf16_scan_product_rounding(dev):
    """T X of the bf16 scan, a product of two f32 operands, one term at a time: k_0 = e_0, k_1 =
    e_0 + e_1, no decay, a zero state and v_1 = 0 leave T[1][0] = -beta_1, X[0] = beta_0 v_0 and
    row 1 of the state = -beta_1 beta_0 v_0, with every other step exact (v_0 powers of
    two).  Bound: twice the f32 rounding of the product.  Half the heads have a leading
    one, zeros and then ones, values of which the six largest products of truncated bf16
    pieces leave out 2^-21."""
    from gguf_runner_amd import ops
    H, d = 64, 128
    rng = np.random.default_rng(8)
    beta = rng.uniform(0.5, 1.0, (2, H)).astype(np.float32)
    beta[:, ::2] = 0.5 + (0xffff - rng.integers(0, 9, (2, H // 2))) * np.float32(2.0 ** -24)
    q, k, v = (np.zeros((2, H, d), np.float32) for _ in range(3))
    k[:, :, 0] = k[1, :, 1] = 1
    v[0] = 2.0 ** (np.arange(d) % 16 - 8)
    st = torch.zeros((H, d, d), device=dev)
    ops.DeltaNetCall(*(torch.from_numpy(x).to(dev).bfloat16() for x in (q, k, v)), torch.zeros((2, H), device=dev),
                     torch.from_numpy(beta).to(dev), st, torch.empty((2, H, d), device=dev), l2norm=False, algo=2)()
    S = st.cpu().numpy().astype(np.float64)
    want = -(beta[0].astype(np.float64) * beta[1])[:, None] * v[0]
    rel = np.abs(S[:, 1] / want - 1).max()
    assert rel <= 2.0 ** -23, np.log2(rel)


def _substitution(A):
    """(I + A)^-1 of strictly lower f32 matrices [n][64][64] by forward substitution in f32, each
    row's sum as chains of four terms summed in a tree."""
    n = A.shape[0]
    X = np.zeros_like(A)
    for t in range(64):
        p = (A[:, t, :, None] * X).reshape(n, 16, 4, 64).astype(np.float32)
        c = ((p[:, :, 0] + p[:, :, 1]) + p[:, :, 2]) + p[:, :, 3]
        while c.shape[1] > 1:
            c = c[:, 0::2] + c[:, 1::2]
        X[:, t] = -c[:, 0]
        X[:, t, t] += np.float32(1)
    return X


@pytest.mark.parametrize("fmt", ["F32", "F16"])
def test_deltanet_prep_inverse_is_as_close_as_substitution(orc, dev, fmt):
    """T = (I + A)^-1 of the prep, read from the workspace's blocks, against 64 bits: at most 1.7
    times as far off as f32 substitution with tree sums (1.45 times with the prep's sums
    done on the CPU; 2.4 times with one chain over each block row's terms).  Keys whose
    products are exact (first element 1, a few of +-1/8), no decay and betas of 8 bits make
    A itself exact; T is then far from I."""
    from gguf_runner_amd import ops
    H, d, T = 8, 128, 512
    rng = np.random.default_rng(21)
    k = rng.integers(-1, 2, (T, H, d)) * (rng.random((T, H, d)) < 0.15) / 8.0
    k[:, :, 0] = 1
    beta = rng.integers(32, 224, (T, H)) / 256.0
    dt = torch.float32 if fmt == "F32" else torch.float16
    row = lambda x: torch.from_numpy(x).to(dev, dt)
    call = ops.DeltaNetCall(row(np.zeros_like(k)), row(k), row(np.zeros_like(k)), torch.zeros((T, H), device=dev),
                            torch.from_numpy(beta.astype(np.float32)).to(dev), torch.zeros((H, d, d), device=dev),
                            torch.empty((T, H, d), device=dev), l2norm=False, algo=2)
    call()
    torch.cuda.synchronize()
    first = -call.ws.data_ptr() % 256 + -(-32 * H // 256) * 256
    blocks = call.ws.cpu().numpy()[first:first + T // 64 * H * 22528].view(np.float32).reshape(T // 64, H, 5632)
    m, c = np.arange(16)[:, None], np.arange(16)[None]
    at = (4 * m + ((c >> 2) ^ ((m >> 2) & 3))) * 4 + (c & 3)
    got = np.zeros((T // 64, H, 64, 64), np.float32)
    for r in range(4):
        for q in range(r + 1):
            got[:, :, 16 * r:16 * r + 16, 16 * q:16 * q + 16] = blocks[:, :, 256 * (r * (r + 1) // 2 + q) + at]
    kk = k.reshape(T // 64, 64, H, d).transpose(0, 2, 1, 3)
    A = np.tril(beta.reshape(T // 64, 64, H).transpose(0, 2, 1)[..., None] * (kk @ kk.transpose(0, 1, 3, 2)), -1)
    assert np.array_equal(A, A.astype(np.float32))
    want = np.linalg.inv(np.eye(64) + A)
    off = lambda x: np.linalg.norm(x - want, axis=(2, 3)) / np.linalg.norm(want, axis=(2, 3))
    sub = _substitution(A.reshape(-1, 64, 64).astype(np.float32)).reshape(want.shape)
    assert off(got).mean() <= 1.7 * off(sub).mean(), (off(got).mean(), off(sub).mean())


@pytest.mark.parametrize("d,algo,fmt_name", [(64, 1, "F32"), (64, 0, "BF16"), (256, 1, "F32"), (256, 2, "F16")])
def test_deltanet_state_sizes_64_and_256(orc, dev, d, algo, fmt_name):
    """State sizes other than 128 (the reference takes any ssm_state_size, math.rs:566):
    the token recurrence at d = 64 and 256, also when the chunked or automatic algorithm
    is asked for (the chunked kernels are built for 128), in two calls that carry the
    state."""
    fmt = getattr(orc, fmt_name)
    got, ref, S, Sref = _run(orc, dev, 150, 3, d, 900 + d + algo, fmt, algo, chunks=[70, 80])
    assert float(np.abs(got - ref).max()) <= TOL
    assert float(np.abs(S - Sref).max()) <= TOL
