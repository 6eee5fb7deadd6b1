"""Config 2 end to end on the GPU: the Qwen3 decoder stack (prefill of the
state head in 512-token chunks, one packed pass of the 512-token tail and 64
question blocks of 48 tokens, code-head readout) against the oracle's
restatement of Qwen3::prefill / forward_packed (qwen3.rs:346-401).

Bars: the answer-code probabilities in f32 to |dp| < 5e-5 (the reference's
end-to-end bar); the final hidden state in f32 to 1e-4 and the cached K/V to
1e-4.  bf16 has no published end-to-end bar: it is reported and held to the
bf16 budget of the hidden state (2e-2 relative).  The full 28-layer config
is compared with a fixture the oracle wrote (tests/golden/make_c2_golden.py):
running the oracle over 1.5e10 FLOP of linear layers takes minutes.
"""
import ctypes as C
import os

import numpy as np
import pytest

from cev_hip import configs
from cev_hip._abi import CEV_LINEAR_WORKSPACE_BYTES, check, lib
from helpers import to_np

pytestmark = pytest.mark.gpu

P_TOL = 5e-5
HID_F32_TOL = 1e-4
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "c2_f32.npz")
GOLDEN_BF16 = os.path.join(os.path.dirname(__file__), "golden", "c2_bf16.npz")
HF_GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "c2_hf_f32.npz")
BF16_P_TOL = 3e-2  # the reference's |dp| bar for non-f32 runs (parity_models.rs:42)


def _say(msg):
    print(msg, flush=True)


def _request(w):
    state, qs, codes = w.ids()
    return (state, list(qs)), codes


def _gpu_engine(w, weights, device, budget=None, pass_tokens=None, capacity=None):
    from cev_hip.engine import DeviceEngine
    from cev_hip.qwen3 import Qwen3Stack
    stack = Qwen3Stack(w, weights, device, capacity=capacity or (w.state_tokens + w.questions * w.q_len))
    _, codes = _request(w)
    return DeviceEngine(stack, budget=budget or w.state_tokens, code_ids=codes, pass_tokens=pass_tokens or w.pass_tokens,
                        prefill_chunk=w.prefill_chunk)


def _gpu_config(w, weights, device):
    """The Qwen3-1.7B-shaped packed-pass flow on the device through the engine (prefill of the
    head into the prefix store's slots, one packed pass of the tail and the
    questions).  Returns (probabilities, hidden, engine)."""
    from cev_hip.qwen3 import softmax64
    eng = _gpu_engine(w, weights, device)
    req, _ = _request(w)
    r = eng.run_many([req])[0]
    assert eng.passes == 1 and not r["prefix_cached"]
    return softmax64(r["logits"]), r["hidden"], eng


def _oracle_engine(w, weights, budget=None, pass_tokens=None):
    from oracle.engine import OracleEngine
    from oracle.qwen3_stack import Qwen3Oracle
    _, codes = _request(w)
    return OracleEngine(Qwen3Oracle(w, weights), budget or w.state_tokens, codes, pass_tokens=pass_tokens or w.pass_tokens,
                        prefill_chunk=w.prefill_chunk)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("rows,hidden,residual", [(3584, 2048, False), (37, 2048, True), (5, 4096, True), (1, 64, False),
                                                  (300, 5120, True), (7, 12288, False)])
def test_layer_norm_vs_oracle(gpu, orc, bf16, rows, hidden, residual):
    """cev_rms_norm_seq (the reference's element-order sum) against the
    oracle's rms_norm bit for bit, and cev_rms_norm (tree-order sum) within
    a few roundings of it: the two sums differ only in their last f32 bits,
    so m moves by at most one step of the model dtype and y by a few (row counts
    that leave a partial workgroup; widths up to and past the wave kernel's
    16 chunks per lane; x_out aliases x as in the stack)."""
    import cev_hip
    from helpers import to_dev
    rng = np.random.default_rng(rows + hidden)
    x = rng.standard_normal((rows, hidden)).astype(np.float32) * 3
    h = rng.standard_normal((rows, hidden)).astype(np.float32)
    w = (1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    if bf16:
        x, h, w = orc.round_bf16(x), orc.round_bf16(h), orc.round_bf16(w)
    xs = (orc.round_bf16(x + h) if bf16 else (x + h)) if residual else x
    want = orc.rms_norm(xs, w, 1e-6, bf16)
    step = 2.0 ** -6 if bf16 else 2.0 ** -16
    for sequential in (True, False):
        dx, dh, dw = to_dev(x, bf16, gpu), to_dev(h, bf16, gpu), to_dev(w, bf16, gpu)
        y = cev_hip.rms_norm(dx, dw, 1e-6, h=dh if residual else None, x_out=dx if residual else None, sequential=sequential)
        got = to_np(y)
        if residual:
            assert np.array_equal(to_np(dx), xs)
        if sequential:
            assert np.array_equal(got, want)
        else:
            err = np.abs(got - want)
            assert np.all(err <= step * np.abs(want) + 1e-30), float((err / np.maximum(np.abs(want), 1e-30)).max())


@pytest.mark.parametrize("bf16", [False, True])
def test_swiglu_matches_oracle(gpu, bf16):
    import cev_hip
    from helpers import to_dev
    from oracle.qwen3_stack import _silu_mul
    rng = np.random.default_rng(3)
    gu = rng.standard_normal((300, 2 * 1024)).astype(np.float32) * 2
    if bf16:
        from oracle import round_bf16
        gu = round_bf16(gu)
    d = to_dev(gu, bf16, gpu)
    out = to_np(cev_hip.swiglu(d[:, :1024], d[:, 1024:]))
    want = _silu_mul(gu[:, :1024], gu[:, 1024:], bf16)
    # exp may differ by an ulp between libm and the device; bf16 then by at most one bf16 step
    tol = 2.0 ** -7 if bf16 else 2e-6
    assert np.all(np.abs(out - want) <= tol * np.maximum(np.abs(want), 1e-3))


@pytest.mark.parametrize("bf16", [False, True])
def test_stack_two_layers_vs_oracle(gpu, orc, bf16):
    """Config 2's widths and token layout at 2 layers and a 4096-token vocab."""
    from oracle.qwen3_stack import softmax64
    w = configs.c2(bf16, n_layers=2, vocab=4096)
    _say(f"test stack: bf16={bf16} layers={w.n_layers} hidden={w.hidden} state={w.state_tokens} pass={w.pass_tokens}")
    weights = w.weights()
    p, hid, eng = _gpu_config(w, weights, gpu)
    oe = _oracle_engine(w, weights)
    req, _ = _request(w)
    r = oe.run_many([req])[0]
    rp, rh = softmax64(r["logits"]), r["hidden"]
    dp = float(np.abs(p - rp).max())
    dh = float(np.abs(hid - rh).max())
    scale = float(np.abs(rh).max())
    # the cached K/V of the prefix after the pass: head (prefill) + tail
    # (kept from the pass), at the slots the store gave it, layer 1
    (begin, n), = eng.store.entries()
    assert n == w.state_tokens
    L1 = eng.stack.layers[1]
    kc, vc = to_np(L1["k"][:, begin: begin + n]), to_np(L1["v"][:, begin: begin + n])
    (_, okv), = oe.cache.entries
    dk = float(np.abs(kc - okv[1][0]).max())
    dv = float(np.abs(vc - okv[1][1]).max())
    _say(f"  |dp| {dp:.3g}  max|dhidden| {dh:.3g} (|hidden| <= {scale:.3g})  cache |dk| {dk:.3g} |dv| {dv:.3g}")
    if bf16:
        assert dh <= 2e-2 * scale and dk <= 2e-2 * float(np.abs(okv[1][0]).max())
    else:
        assert dp < P_TOL
        assert dh <= HID_F32_TOL and dk <= HID_F32_TOL and dv <= HID_F32_TOL


def test_stack_second_pass_reads_the_cached_prefix(gpu, orc):
    """A later request on the same state: the whole state is a store hit (no
    prefill, no tail) and new questions attend to the slots the first call
    left behind."""
    from oracle.qwen3_stack import softmax64
    w = configs.c2(False, n_layers=2, vocab=4096, questions=8)
    weights = w.weights()
    _, _, eng = _gpu_config(w, weights, gpu)
    oe = _oracle_engine(w, weights)
    (state, qs), _ = _request(w)
    oe.run_many([(state, qs)])
    q2 = [q[::-1].copy() for q in qs]
    r = eng.run_many([(state, q2)])[0]
    ro = oe.run_many([(state, q2)])[0]
    assert r["prefix_cached"] and ro["prefix_cached"]
    dp = float(np.abs(softmax64(r["logits"]) - softmax64(ro["logits"])).max())
    _say(f"test second pass: |dp| {dp:.3g}, max|dhidden| {float(np.abs(r['hidden'] - ro['hidden']).max()):.3g}")
    assert dp < P_TOL


def test_engine_request_and_twin_then_eviction(gpu, orc):
    """Row f2: a request and its content-free calibration twin (two plans,
    two tails) in one call, split into passes by the token budget,
    through the device prefix store (the first call needs more than one
    pass under the 1000-token budget); then a second call where the request's
    prefix is a hit and a new twin's put evicts the first twin (LRU by
    tokens).  f32 probabilities against the oracle engine at |dp| < 5e-5,
    and the store's entries against the oracle's PrefixCache."""
    from oracle.qwen3_stack import softmax64
    w = configs.c2(False, n_layers=2, vocab=4096, questions=6, q_len=20)
    weights = w.weights()
    rng = np.random.default_rng(12)
    qs = [rng.integers(0, w.vocab, int(rng.integers(8, 30))) for _ in range(6)]
    req = (rng.integers(0, w.vocab, 1100), qs)
    twin = (rng.integers(0, w.vocab, 300), qs)
    twin2 = (rng.integers(0, w.vocab, 420), qs)
    budget = 1100 + 300 + 420 - 1
    eng = _gpu_engine(w, weights, gpu, budget=budget, pass_tokens=1000, capacity=4096)
    oe = _oracle_engine(w, weights, budget=budget, pass_tokens=1000)
    worst = 0.0
    passes = []
    for call, reqs in enumerate(([req, twin], [req, twin2])):
        got = eng.run_many(reqs)
        passes.append(eng.passes)
        want = oe.run_many(reqs)
        for g, r in zip(got, want):
            assert g["prefix_cached"] == r["prefix_cached"]
            worst = max(worst, float(np.abs(softmax64(g["logits"]) - softmax64(r["logits"])).max()))
        lens = [n for _, n in eng.store.entries()]
        assert lens == [len(k) for k, _ in oe.cache.entries], (call, lens)
        _say(f"call {call}: cached={[g['prefix_cached'] for g in got]} entries={lens} passes={eng.passes} |dp| {worst:.3g}")
    assert eng.passes == oe.passes and passes[0] >= 2
    assert [len(k) for k, _ in oe.cache.entries] == [1100, 420]  # the first twin was evicted
    assert worst < P_TOL


@pytest.mark.skipif(not os.path.exists(HF_GOLDEN), reason="tests/golden/c2_hf_f32.npz not generated")
def test_stack_two_layers_vs_hf_transformers(gpu):
    """The device engine against HF transformers' Qwen3ForCausalLM asked
    each question alone over [state || question] (tests/golden/make_c2_hf.py),
    the Qwen3-1.7B-shaped widths at 2 layers, f32: the reference's own bar
    (README.md:48)."""
    from cev_hip.qwen3 import softmax64
    g = np.load(HF_GOLDEN)
    w = configs.c2(False, n_layers=int(g["layers"]), vocab=int(g["vocab"]), questions=int(g["questions"]))
    p, hid, _ = _gpu_config(w, w.weights(), gpu)
    dp = float(np.abs(p - g["p"]).max())
    dh = float(np.abs(hid - g["hidden"]).max())
    _say(f"stack vs HF transformers: |dp| {dp:.3g}  max|dhidden| {dh:.3g}")
    assert dp < P_TOL and dh < 1e-3


@pytest.mark.skipif(not os.path.exists(GOLDEN_BF16), reason="tests/golden/c2_bf16.npz not generated")
def test_config2_full_bf16_vs_golden(gpu):
    """All 28 layers and the full vocab in bf16 (the config's own dtype)
    against the oracle's bf16 fixture: |dp| <= 3e-2, the bar the reference
    holds its own non-f32 runs to (parity_models.rs:42).  The hidden state
    is reported and held to 7 % of its norm (relative RMS): the device
    keeps attention scores in f32 where candle rounds them to bf16, and
    rounds f32 GEMM sums taken in another order, so every layer moves some
    elements by a bf16 step and 28 residual layers accumulate it (about
    1.4 % at 2 layers; 4.57 % at 28, with |dp| 0.024)."""
    w = configs.c2(True)
    g = np.load(GOLDEN_BF16)
    _say(f"test 28-layer stack bf16: layers={w.n_layers} vocab={w.vocab}")
    p, hid, _ = _gpu_config(w, w.weights(), gpu)
    dp = float(np.abs(p - g["p"]).max())
    dh = float(np.abs(hid - g["hidden"]).max())
    rel = float(np.linalg.norm(hid - g["hidden"]) / np.linalg.norm(g["hidden"]))
    scale = float(np.abs(g["hidden"]).max())
    _say(f"  |dp| {dp:.3g}  hidden relative RMS {rel:.3g}, max|dhidden| {dh:.3g} (|hidden| <= {scale:.3g})")
    assert dp <= BF16_P_TOL and rel <= 0.07


@pytest.mark.skipif(not os.path.exists(GOLDEN), reason="tests/golden/c2_f32.npz not generated")
def test_config2_full_f32_vs_golden(gpu):
    """All 28 layers and the full vocab, f32: probabilities against the
    oracle's fixture."""
    w = configs.c2(False)
    g = np.load(GOLDEN)
    _say(f"test 28-layer stack f32: layers={w.n_layers} vocab={w.vocab} (weights {w.n_layers * 201 + 1245} MB f32)")
    p, hid, _ = _gpu_config(w, w.weights(), gpu)
    dp = float(np.abs(p - g["p"]).max())
    dh = float(np.abs(hid - g["hidden"]).max())
    _say(f"  |dp| {dp:.3g}  max|dhidden| {dh:.3g}")
    assert dp < P_TOL


def _debias_inputs(rng, ks, max_perm=4, invariant=False):
    from oracle.qwen3_stack import rotated_order, rotation_shifts
    ld = max(ks)
    rows, orders, begin, length = [], [], [], []
    for k in ks:
        f = rng.standard_normal(k).astype(np.float32) * 3
        begin.append(len(rows))
        shifts = rotation_shifts(k, max_perm)
        length.append(len(shifts))
        base = list(rng.permutation(k))
        for s in shifts:
            order = rotated_order(base, s)
            row = rng.standard_normal(ld).astype(np.float32) * 3
            if invariant:
                row[:k] = f[order]
            rows.append(row)
            orders.append(order + [0] * (ld - k))
    return (np.array(rows), np.array(orders, np.int32), np.array(begin, np.int32), np.array(length, np.int32),
            np.array(ks, np.int32))


def _device_debias(gpu, logits, order, begin, length, ks, calib=None):
    import torch
    import cev_hip
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(gpu)
    out = cev_hip.debias_scores(t(logits), t(order), t(begin), t(length), t(ks), calib=None if calib is None else t(calib))
    torch.cuda.synchronize()
    return to_np(out)


@pytest.mark.parametrize("calibrated", [False, True])
def test_debias_scores_match_oracle(gpu, calibrated):
    """cev_debias_scores against the oracle's restatement of
    Service::run_debiased's averaging (service.rs:330-345): the packed pass's
    16 questions x 4 rotations x 8 codes plus ragged option counts (1..64).
    f64 exp / log may differ by an ulp between libm and the device: the f32
    scores are held to 2 ulp-scale."""
    from oracle.qwen3_stack import debias_scores
    rng = np.random.default_rng(21 + calibrated)
    ks = [8] * 16 + [2, 3, 5, 7, 1, 64, 13]
    logits, order, begin, length, kk = _debias_inputs(rng, ks)
    calib = rng.standard_normal(logits.shape).astype(np.float32) * 2 if calibrated else None
    got = _device_debias(gpu, logits, order, begin, length, kk, calib)
    want = debias_scores(logits, order, begin, length, kk, calib=calib)
    for q, k in enumerate(ks):
        d = np.abs(got[q, :k] - want[q, :k])
        assert np.all(d <= 2.5e-7 * np.maximum(np.abs(want[q, :k]), 1.0)), (q, k, d.max())
    _say(f"debias calibrated={calibrated}: {len(ks)} questions, max|d| {max(np.abs(got[q, :k] - want[q, :k]).max() for q, k in enumerate(ks)):.3g}")


def test_debias_position_invariant_model_and_invalid_spans(gpu):
    """The reference's own property (runtime.rs:185-207): averaging the
    rotations of a position-invariant model gives each option its plain
    log-probability.  Spans outside the variants, an option count of 0 and
    an order that is not a permutation give NaN rows."""
    from oracle.qwen3_stack import log_softmax64
    rng = np.random.default_rng(9)
    ks = [5, 2, 8]
    logits, order, begin, length, kk = _debias_inputs(rng, ks, invariant=True)
    got = _device_debias(gpu, logits, order, begin, length, kk)
    for q, k in enumerate(ks):
        # option o's logit is the same wherever it is shown: read it off variant 0
        canon = np.empty(k, np.float32)
        canon[order[begin[q], :k]] = logits[begin[q], :k]
        assert np.allclose(got[q, :k], log_softmax64(canon), rtol=0, atol=2e-6)
    bad_begin = np.array([0, len(logits) - 1, 0], np.int32)
    bad_len = np.array([len(logits) + 1, 2, 1], np.int32)
    bad_k = np.array([5, 2, 0], np.int32)
    got = _device_debias(gpu, logits, order, bad_begin, bad_len, bad_k)
    assert np.isnan(got).all()
    broken = order.copy()
    broken[begin[1], 0] = 2  # k = 2: option index out of range
    got = _device_debias(gpu, logits, broken, begin, length, kk)
    assert np.isnan(got[1, :2]).all() and np.isfinite(got[0, :5]).all() and np.isfinite(got[2, :8]).all()
    # a repeated index (every entry in range, option 1 never named) is not a
    # permutation either
    dup = order.copy()
    dup[begin[2] + 1, :8] = [0, 0, 2, 3, 4, 5, 6, 7]
    got = _device_debias(gpu, logits, dup, begin, length, kk)
    assert np.isnan(got[2, :8]).all() and np.isfinite(got[0, :5]).all() and np.isfinite(got[1, :2]).all()


@pytest.mark.parametrize("m,n,k,parts", [(128, 12288, 2048, 2), (700, 2052, 2044, 2), (200, 3000, 6140, 4), (200, 12288, 36, 1),
                                         (912, 2048, 6144, 2), (1000, 4095, 516, 1), (2050, 4096, 128, 1), (1300, 2048, 2048, 1)])
def test_split_f32_product(gpu, m, n, k, parts):
    """f32 products on the bf16 matrix cores: remainders of the 128-wide tiles
    and of the 32-deep slices, in one part of k and in several (k = 36: two
    slices, most loads past the end), against f64.
    Each value: the first parts' sum is rounded once per 16 of the k products
    and in a few more adds, 2^-24 each of at most sum |x| |w|; the accumulators
    of 16 products may round inside (factor 2); the dropped part products add
    2^-24.
    The norm: N = k / 16 roundings of partial sums that grow like a random
    walk, each uniform in +-2^-24 of a sum, are 2^-24 sqrt(N / 6) of the result
    (measured: 2.7e-7 at k = 2048, 4.9e-7 at 6144), with 40 % and one more
    rounding to spare.  Without any one of the six part products it is 2.4e-6,
    with one accumulator for all of them 7e-7 and 1.2e-6."""
    import torch

    import cev_hip
    form = C.c_int32()
    check(lib().cev_linear_form(cev_hip.CEV_F32, m, n, k, CEV_LINEAR_WORKSPACE_BYTES, C.byref(form)))
    assert form.value == parts
    g = torch.Generator().manual_seed(m + k)
    x, w = torch.randn(m, k, generator=g).to(gpu), torch.randn(n, k, generator=g).to(gpu)
    ld = n + 4 - n % 4 if n % 4 else n
    out = torch.full((m, ld), float("nan"), device=gpu)[:, :n]
    got = cev_hip.linear(x, w, out=out, alpha=0.5).double()
    want = 0.5 * x.double() @ w.double().t().contiguous()
    bound = 0.5 * (2 * (k / 16 + 16) + 1) * 2.0**-24 * (x.double().abs() @ w.double().abs().t().contiguous())
    assert ((got - want).abs() <= bound).all()
    rel = float((got - want).norm() / want.norm())
    print(f"split f32 product {m} x {n} x {k}: error {rel:.3g}", flush=True)
    assert rel <= 1.4 * 2.0**-24 * ((k / 96) ** 0.5 + 1)


def test_products_on_two_streams_do_not_share_sums(gpu):
    """f32 products whose parts of k are summed through a workspace, queued on
    two streams at once, with and without a current stream: each call has a
    workspace of its own stream's."""
    import torch

    import cev_hip
    m, n, k = 912, 2048, 6144
    g = torch.Generator().manual_seed(12)
    x = [torch.randn(m, k, generator=g).to(gpu) for _ in range(2)]
    w = torch.randn(n, k, generator=g).to(gpu)
    want = [cev_hip.linear(v, w) for v in x]
    streams = [torch.cuda.Stream() for _ in range(2)]
    out = [[torch.empty_like(want[0]) for _ in range(8)] for _ in range(2)]
    torch.cuda.synchronize()
    for i in range(8):
        for j in range(2):
            if i % 2:
                cev_hip.linear(x[j], w, out=out[j][i], stream=streams[j])
            else:
                with torch.cuda.stream(streams[j]):
                    cev_hip.linear(x[j], w, out=out[j][i])
    torch.cuda.synchronize()
    for j in range(2):
        assert all(torch.equal(o, want[j]) for o in out[j])


def test_split_f32_product_keeps_infinities(gpu):
    """Values without bf16 parts (infinite, or above bf16's range) give what
    plain f32 products give: their tile is computed again one by one."""
    import torch

    import cev_hip
    m, n, k = 256, 12288, 64
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    x[3, 5], x[40, 7], x[200, 0], w[900, 9] = float("inf"), 3.4e38, float("nan"), -float("inf")
    w[:, 7] = 1e-30
    got = cev_hip.linear(x.to(gpu), w.to(gpu)).cpu()
    want = x.double() @ w.double().t()
    fin = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), fin)
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)].float())
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.allclose(got[fin].double(), want[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dt,odt", [("bf16", "bf16"), ("bf16", "f32"), ("f32", "bf16"), ("f32", "f32")])
@pytest.mark.parametrize("width,off", [(8, 0), (2048, 0), (2056, 0), (2048, 1), (12, 0), (7, 0)])
def test_gather_rows_forms(gpu, dt, odt, width, off):
    """Wide and element-wise gathers (odd widths, unaligned views) give the
    same rows, and an index outside the table a NaN row."""
    import torch

    import cev_hip
    T, O = (torch.bfloat16 if d == "bf16" else torch.float32 for d in (dt, odt))
    base = torch.randn(50, width + off, generator=torch.Generator().manual_seed(width)).to(T).to(gpu)
    table = base[:, off:]
    ids = torch.tensor([0, 49, 7, -1, 50, 7], dtype=torch.int32, device=gpu)
    got = cev_hip.gather_rows(table, ids, out_dtype=O)
    want = table[[0, 49, 7, 0, 0, 7]].to(O)
    assert torch.equal(got[[0, 1, 2, 5]], want[[0, 1, 2, 5]])
    assert got[3:5].isnan().all()
    assert torch.equal(cev_hip.gather_rows(table, out_dtype=O), table.to(O))
