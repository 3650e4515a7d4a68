"""GPU: the MATH attention backend (ythip_attn_math), masked matmul
(ythip_gemm_masked), predicate / diagonal masks and strided or broadcast K/V
on the flash path, against the oracle's restatements (pinned to the reference
in test_oracle_math.py).

Bars: fp32 max|g - r| <= 1e-4 * max|r| (attention outputs: 1e-4 absolute on
O(1) values); bf16 / fp16 the 2e-2 / MAE 1e-3 bar of check16, with the oracle
run on the same 16-bit-rounded inputs."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import check16

pytestmark = pytest.mark.gpu


def _t(x, dev, dt=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dev).to(dt)


def _f(t):
    return t.float().cpu().numpy()


def _ref_heads(orc, Q, K, V, kw, backend):
    """Q [H, Lq, D] etc. -> oracle output, MATH restatement or flash."""
    if backend == "math":
        return orc.sdpa_math(Q, K, V, 0.0, **kw)
    mask, diag, bias = kw.get("mask"), kw.get("diag"), kw.get("bias")
    Lq, Lkv = Q.shape[1], K.shape[1]
    if diag is not None:
        mask = np.arange(Lkv)[None, :] <= np.arange(Lq)[:, None] + diag
    return np.stack([orc.flash_attention(Q[h], K[h], V[h], 1 / np.sqrt(np.float32(Q.shape[2])), mask, bias)
                     for h in range(Q.shape[0])])


def _mask_arg(kw, Lq, Lkv):
    if "diag" in kw:
        return ("diag", kw["diag"])
    if "pred" in kw:
        off = kw["pred"]
        return lambda i, j: j <= i + off
    return kw.get("mask_t")


CASES = [  # (H, Lq, Lkv, D, Dv, mask form)
    (2, 7, 9, 16, 16, None),
    (3, 40, 70, 64, 64, "bool"),
    (2, 64, 64, 128, 128, "causal"),
    (2, 33, 50, 64, 32, "diag5"),
    (1, 20, 20, 32, 32, "pred0"),
    (2, 16, 24, 64, 64, "bool_bias"),
    (1, 9, 9, 8, 8, "diag-3"),
]


def _case(orc, case, seed):
    H, Lq, Lkv, D, Dv, form = case
    rng = np.random.default_rng(seed)
    Q = rng.standard_normal((H, Lq, D)).astype(np.float32)
    K = rng.standard_normal((H, Lkv, D)).astype(np.float32)
    V = rng.standard_normal((H, Lkv, Dv)).astype(np.float32)
    kw, arg = {}, {}
    if form in ("bool", "bool_bias"):
        m = rng.random((Lq, Lkv)) < 0.6
        m[1] = False
        kw["mask"] = m
        arg["mask_t"] = torch.from_numpy(m)
        if form == "bool_bias":
            b = rng.standard_normal((Lq, Lkv)).astype(np.float32)
            kw["bias"] = b
            arg["bias"] = b
    elif form == "causal":
        kw["diag"] = Lkv - Lq
        arg["causal"] = True
    elif form is not None and form.startswith("diag"):
        kw["diag"] = int(form[4:])
        arg["diag"] = kw["diag"]
    elif form is not None and form.startswith("pred"):
        kw["diag"] = int(form[4:])
        arg["pred"] = kw["diag"]
    return Q, K, V, kw, arg


@pytest.mark.parametrize("backend", ["math", "flash"])
@pytest.mark.parametrize("case", CASES)
def test_sdpa_backends_fp32_vs_oracle(orc, yt, dev, backend, case):
    Q, K, V, kw, arg = _case(orc, case, 5)
    mask = "causal" if arg.get("causal") else _mask_arg(arg, Q.shape[1], K.shape[1])
    bias = _t(arg["bias"], dev) if "bias" in arg else None
    got = yt.scaled_dot_product_attention(_t(Q, dev), _t(K, dev), _t(V, dev), 0.0, mask=mask, bias=bias,
                                          backend=backend)
    torch.cuda.synchronize()
    ref = _ref_heads(orc, Q, K, V, kw, backend)
    assert np.abs(_f(got) - ref).max() <= 1e-4, (backend, case)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [CASES[1], CASES[2], CASES[3], CASES[5]])
def test_sdpa_math_16bit_vs_oracle(orc, yt, dev, dt, case):
    Q, K, V, kw, arg = _case(orc, case, 6)
    rnd = (lambda x: orc.bf16_to_f32(orc.bf16_round(x))) if dt == torch.bfloat16 else \
        (lambda x: orc.f16_to_f32(orc.f16_round(x)))
    Q, K, V = rnd(Q), rnd(K), rnd(V)
    mask = "causal" if arg.get("causal") else _mask_arg(arg, Q.shape[1], K.shape[1])
    bias = _t(arg["bias"], dev) if "bias" in arg else None
    got = yt.scaled_dot_product_attention(_t(Q, dev, dt), _t(K, dev, dt), _t(V, dev, dt), 0.0, mask=mask,
                                          bias=bias, backend="math")
    torch.cuda.synchronize()
    ref = orc.sdpa_math(Q, K, V, 0.0, **kw)
    check16(orc, _f(got), ref, "bf16" if dt == torch.bfloat16 else "f16", True, f"math {case}")


@pytest.mark.parametrize("backend", ["math", "flash"])
def test_ymodel2_pega2_layout(orc, yt, dev, backend):
    """The ymodel2 example's attention (example/ymodel2-s-2/ymodel2.cpp:188-262):
    q [b, 2, hh, l, hd]; k = repeat_kv of a [b, 2, L, hd] cache (0-stride over
    hh); v = the cache's second half repeated over the first axis (0-stride);
    the cache stored transposed ([b, 2, hd, L], read through .transpose) and a
    ring-wrapped bool causal mask."""
    rng = np.random.default_rng(8)
    b, hh, l, L, hd = 2, 4, 5, 23, 64
    q = rng.standard_normal((b, 2, hh, l, hd)).astype(np.float32)
    cache_t = rng.standard_normal((b, 2, hd, L)).astype(np.float32)  # transposed storage
    wp = 7  # ring write position: logical order starts at wp
    mask = np.zeros((l, L), bool)
    for qi in range(l):
        for ki in range(L):
            mask[qi, ki] = (ki - wp + L) % L <= L - l + qi
    kvc = torch.from_numpy(cache_t).to(dev)
    kv = kvc.transpose(-1, -2)                          # [b, 2, L, hd], d-stride L
    k5 = kv.unsqueeze(2).expand(b, 2, hh, L, hd)        # repeat_kv: 0-stride over hh
    v5 = kv[:, 1:2].expand(b, 2, L, hd).unsqueeze(2).expand(b, 2, hh, L, hd)
    out = yt.scaled_dot_product_attention(_t(q, dev), k5, v5, 0.125, mask=torch.from_numpy(mask), backend=backend)
    torch.cuda.synchronize()
    kv_np = np.swapaxes(cache_t, -1, -2)
    for bi in range(b):
        for s in range(2):
            for j in range(hh):
                K = kv_np[bi, s][None]
                Vv = kv_np[bi, 1][None]
                if backend == "math":
                    ref = orc.sdpa_math(q[bi, s, j][None], K, Vv, 0.125, mask=mask)[0]
                else:
                    ref = orc.flash_attention(q[bi, s, j], K[0], Vv[0], 0.125, mask)
                assert np.abs(_f(out[bi, s, j]) - ref).max() <= 1e-4


def test_flash_transposed_keys_decode_and_prefill(orc, yt, dev):
    """K and V stored [B, H, D, L] (d-major) on the flash path: the row-wise
    kernel reads them through their strides (the reference copies to contiguous
    for q_len > 1 and reads strided for q_len == 1, ops.inl:176-189)."""
    rng = np.random.default_rng(9)
    B, H, L, D = 1, 2, 300, 64
    kt = rng.standard_normal((B, H, D, L)).astype(np.float32)
    vt = rng.standard_normal((B, H, D, L)).astype(np.float32)
    for Lq in (1, 17):
        q = rng.standard_normal((B, H, Lq, D)).astype(np.float32)
        kd, vd = _t(kt, dev), _t(vt, dev)
        out = yt.scaled_dot_product_attention(_t(q, dev), kd.transpose(-1, -2), vd.transpose(-1, -2), 0.0,
                                              mask="causal")
        torch.cuda.synchronize()
        K, V = np.swapaxes(kt, -1, -2)[0], np.swapaxes(vt, -1, -2)[0]
        ref = orc.sdpa_math(q[0], K, V, 0.0, diag=L - Lq)
        assert np.abs(_f(out[0]) - ref).max() <= 1e-4


def test_flash_diag_masks_on_mfma_path_bf16(orc, yt, dev):
    """Diagonal offsets on the 16-bit MFMA kernel (offset 0 on a rectangular
    problem, negative offsets with rows that see no key)."""
    rng = np.random.default_rng(10)
    H, Lq, Lkv, D = 2, 200, 300, 128
    rnd = lambda x: orc.bf16_to_f32(orc.bf16_round(x))  # noqa: E731
    Q = rnd(rng.standard_normal((H, Lq, D)).astype(np.float32))
    K = rnd(rng.standard_normal((H, Lkv, D)).astype(np.float32))
    V = rnd(rng.standard_normal((H, Lkv, D)).astype(np.float32))
    for off in (0, -40, 150, 10000, -10000):
        got = yt.scaled_dot_product_attention(_t(Q, dev, torch.bfloat16)[None], _t(K, dev, torch.bfloat16)[None],
                                              _t(V, dev, torch.bfloat16)[None], 0.0, mask=("diag", off))
        torch.cuda.synchronize()
        ref = orc.sdpa_math(Q, K, V, 0.0, diag=off)
        check16(orc, _f(got[0]), ref, "bf16", True, f"diag {off}")
        if off <= -Lq:
            assert torch.count_nonzero(got) == 0


@pytest.mark.parametrize("m,n,k", [(13, 17, 32), (256, 384, 128), (1000, 520, 64), (3, 4096, 256)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (0.5, 2.0)])
def test_gemm_masked_fp32(orc, yt, dev, m, n, k, alpha, beta):
    rng = np.random.default_rng(m + n + k)
    A = rng.standard_normal((m, k)).astype(np.float32)
    B = rng.standard_normal((k, n)).astype(np.float32)
    C = rng.standard_normal((m, n)).astype(np.float32)
    mask = rng.random((m, n)) < 0.5
    out = _t(C, dev)
    yt.gemm_masked(_t(A, dev), _t(B, dev), out, torch.from_numpy(mask), alpha, beta)
    torch.cuda.synchronize()
    ref = orc.sgemm_masked(A, B, C.copy(), mask, alpha, beta)
    got = _f(out)
    assert np.array_equal(got[~mask], C[~mask])
    assert np.abs(got - ref).max() <= 1e-4 * np.abs(ref).max()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_masked_matmul_16bit_batched_predicates(orc, yt, dev, dt):
    rng = np.random.default_rng(12)
    bt, m, n, k = 3, 96, 130, 64
    rnd = (lambda x: orc.bf16_to_f32(orc.bf16_round(x))) if dt == torch.bfloat16 else \
        (lambda x: orc.f16_to_f32(orc.f16_round(x)))
    A = rnd(rng.standard_normal((bt, m, k)).astype(np.float32))
    B = rnd(rng.standard_normal((k, n)).astype(np.float32))
    for mask, diag in ((None, 3), (lambda i, j: (i + j) % 3 != 0, None), ("causal", n - m)):
        got = yt.masked_matmul(_t(A, dev, dt), _t(B, dev, dt), mask if mask is not None else ("diag", diag),
                               masked_value=-8192.0)
        torch.cuda.synchronize()
        if callable(mask):
            mk = np.fromfunction(lambda i, j: (i + j) % 3 != 0, (m, n), dtype=int)
            refs = [orc.masked_matmul(A[i], B, mask=mk, value=-8192.0) for i in range(bt)]
        else:
            refs = [orc.masked_matmul(A[i], B, diag=diag, value=-8192.0) for i in range(bt)]
        ref = np.stack(refs)
        vis = ref != -8192.0
        g = _f(got)
        assert np.all(g[~vis] == -8192.0)
        check16(orc, g[vis], ref[vis], "bf16" if dt == torch.bfloat16 else "f16", True, f"masked {mask}")


def test_math_edge_cases(yt, dev):
    q = torch.randn(1, 2, 4, 16, device=dev)
    k = torch.randn(1, 2, 0, 16, device=dev)
    v = torch.randn(1, 2, 0, 8, device=dev)
    out = yt.scaled_dot_product_attention(q, k, v, backend="math")
    torch.cuda.synchronize()
    assert out.shape == (1, 2, 4, 8) and torch.count_nonzero(out) == 0
    with pytest.raises(ValueError):
        yt.scaled_dot_product_attention(q, k, v, backend="eigen")
    k = torch.randn(1, 2, 6, 16, device=dev)
    v = torch.randn(1, 2, 6, 8, device=dev)
    with pytest.raises(ValueError):
        yt.scaled_dot_product_attention(q, k, v, mask=torch.ones(3, 6, dtype=torch.bool), backend="math")


@pytest.mark.parametrize("Lkv", [1500, 4096, 5000])
def test_math_long_rows(orc, yt, dev, Lkv):
    """Rows of up to 1024 / 4096 keys are read once into registers; longer
    rows take the three-pass softmax. Both against the oracle."""
    rng = np.random.default_rng(Lkv)
    H, Lq, D = 2, 8, 64
    Q = rng.standard_normal((H, Lq, D)).astype(np.float32)
    K = rng.standard_normal((H, Lkv, D)).astype(np.float32)
    V = rng.standard_normal((H, Lkv, D)).astype(np.float32)
    m = rng.random((Lq, Lkv)) < 0.5
    m[3] = False
    b = rng.standard_normal((Lq, Lkv)).astype(np.float32)
    got = yt.scaled_dot_product_attention(_t(Q, dev), _t(K, dev), _t(V, dev), 0.0, mask=torch.from_numpy(m),
                                          bias=_t(b, dev), backend="math")
    torch.cuda.synchronize()
    ref = orc.sdpa_math(Q, K, V, 0.0, mask=m, bias=b)
    assert np.abs(_f(got) - ref).max() <= 1e-4
    assert torch.count_nonzero(got[:, 3]) == 0


def _math64(q, k, v, scale, vis, bias):
    """The MATH backend in float64: hidden scores are -1e9 before scale and bias and
    stay in the softmax; rows that see no key are zero when a mask is given."""
    G = q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(G, 0).double(), v.repeat_interleave(G, 0).double()
    s = torch.matmul(q.double(), k.transpose(-1, -2).contiguous())
    if vis is not None:
        s = s.masked_fill(~vis, -1e9)
    s = s * scale
    if bias is not None:
        s = s + bias.double()
    o = torch.matmul(torch.softmax(s, -1), v)
    return o if vis is None else o.masked_fill(~vis.any(-1)[:, None], 0.0)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv", [(1, 1), (5, 63), (64, 65), (65, 129), (130, 256), (300, 333), (2100, 200)])
def test_sdpa_math_one_launch(yt, dev, Sq, Skv, D, dt):
    """The one-launch MATH kernels against float64 at the edges of their 64-query and
    64- / 128-key blocks, every mask kind, GQA 2:1. Beside ordinary scales: a
    negative one and one of 1e-8 (hidden keys keep weight), a bias that lifts
    hidden keys back up (at a scale of 2^-20, where -1e9 scale is exact in fp32 and cancels
    exactly against a bias of 1e9 scale plus eighths). Bound: 32-bit arithmetic on scores up
    to 8 (1e-5 of the values' size) and in 16 bits the rounding of the weights and the result."""
    g = torch.Generator(device=dev).manual_seed(Sq + Skv + D)
    q = torch.randn(2, 4, Sq, D, device=dev, generator=g).to(dt)
    k = torch.randn(2, 2, Skv, D, device=dev, generator=g).to(dt)
    v = torch.randn(2, 2, Skv, D, device=dev, generator=g).to(dt)
    i, j = torch.arange(Sq, device=dev)[:, None], torch.arange(Skv, device=dev)[None, :]
    drop = torch.rand(Sq, Skv, device=dev, generator=g) < 0.4
    drop[Sq // 2] = True
    bias = torch.randn(Sq, Skv, device=dev, generator=g)
    eighths = torch.randint(-16, 17, (Sq, Skv), device=dev, generator=g).float() / 8
    lift = torch.where(drop, 1e9 * 2.0 ** -20 + eighths, bias)
    assert torch.equal(lift.double()[drop], (1e9 * 2.0 ** -20 + eighths.double())[drop])
    cases = [(None, None, 0.0, None), ("causal", j <= i + Skv - Sq, 0.0, None), (("diag", -3), j <= i - 3, 0.0, None),
             (~drop, ~drop, 0.0, None), (~drop, ~drop, 0.0, bias), ("causal", j <= i + Skv - Sq, 1e-8, None),
             (~drop, ~drop, -1e-9, None), (~drop, ~drop, 2.0 ** -20, lift)]
    ulp = {torch.float32: 2e-7, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dt]
    for mask, vis, scale, bs in cases:
        out = yt.scaled_dot_product_attention(q, k, v, scale, mask=mask, bias=bs, backend="math")
        for b in range(2):
            want = _math64(q[b], k[b], v[b], scale or 1.0 / D ** 0.5, vis, bs)
            top = float(v.double().abs().max())
            bound = (1e-5 + ulp) * top + 2 * ulp * want.abs()
            assert ((out[b].double() - want).abs() <= bound).all(), (scale, bs is not None)
        assert torch.isfinite(out).all()
    if Skv >= 63 and Sq > 1:
        # 0 . V as in the product: a non-finite V row behind the mask reaches every row
        v2 = v.clone()
        v2[:, :, Skv - 1, 3] = float("nan")
        out = yt.scaled_dot_product_attention(q, k, v2, mask=("diag", 0), backend="math")
        assert out[..., 3].isnan().all() and torch.isfinite(out[..., :3]).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["NN", "NT", "odd", "c_cols"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (5, 7, 3), (64, 64, 64), (130, 200, 72), (200, 136, 40), (257, 129, 100), (2048, 2056, 40)])
def test_gemm_masked_layouts(yt, dev, m, n, k, layout, dt):
    """The masked store of every product kernel (16-byte aligned rows NN / NT, odd
    rows, a column-major C; 64- and 128-wide tiles, ragged edges): diagonals that
    hide whole tiles, cut them and hide nothing, and bytes; kept or filled; alpha /
    beta. Against float64: (k + 2) 2^-24 sum|a||b| plus the rounding of the result;
    hidden entries exactly."""
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    pad = 1 if layout == "odd" else 0
    A = torch.randn(2, m, k + pad, device=dev, generator=g).to(dt)[:, :, pad:]
    B = torch.randn(2, n, k, device=dev, generator=g).to(dt).transpose(1, 2) if layout == "NT" else \
        torch.randn(2, k, n + pad, device=dev, generator=g).to(dt)[:, :, pad:]
    prod = torch.matmul(A.double(), B.double().contiguous())
    mass = torch.matmul(A.double().abs(), B.double().abs().contiguous())
    i, j = torch.arange(m, device=dev)[:, None], torch.arange(n, device=dev)[None, :]
    bytes_ = torch.rand(m, n, device=dev, generator=g) < 0.5
    ulp = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[dt]
    for mask, vis in [("causal", j <= i + n - m), (("diag", -70), j <= i - 70), (("diag", n), j <= i + n), (bytes_, bytes_)]:
        for alpha, beta, fill in [(1.0, 0.0, -3.0), (1.0, 0.0, None), (0.5, 2.0, 7.0), (0.5, 2.0, None)]:
            C = torch.randn(2, n, m, device=dev, generator=g).to(dt).transpose(1, 2) if layout == "c_cols" else \
                torch.randn(2, m, n + pad, device=dev, generator=g).to(dt)[:, :, pad:]
            C0 = C.double()
            yt.gemm_masked(A, B, C, mask, alpha, beta, fill)
            want = alpha * prod + beta * C0
            bound = (k + 2) * 2.0 ** -24 * mass + ulp * want.abs() + 4 * 2.0 ** -23 * C0.abs() + 1e-7
            ok = (C.double() - want).abs() <= bound  # (false for a NaN)
            assert ok[vis.expand(2, m, n)].all(), (mask if isinstance(mask, (str, tuple)) else "bytes", alpha, fill)
            hid = (~vis).expand(2, m, n)
            assert torch.equal(C.double()[hid], (C0 if fill is None else torch.full_like(C0, fill))[hid])


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("where", ["q", "k", "k_shifted", "apart_in_one_buffer"])
def test_sdpa_math_output_over_an_input(yt, dev, where, dt):
    """O over Q or K (whole, or shifted by some rows) gives the result of an O apart from
    them: one launch would write O while other workgroups read K. Bound: the rounding
    of weights and result (the overlapped call runs in separate launches)."""
    g = torch.Generator(device=dev).manual_seed(5)
    H, S, D = 16, 1024, 64
    buf = torch.randn(4 * H * S * D, device=dev, generator=g).to(dt)
    n = H * S * D
    q, k, v = (buf[i * n:(i + 1) * n].view(1, H, S, D) for i in range(3))
    want = yt.scaled_dot_product_attention(q, k, v, mask="causal", backend="math").double()
    at = {"q": 0, "k": n, "k_shifted": n // 2 + 8 * D, "apart_in_one_buffer": 3 * n}[where]
    out = buf[at:at + n].view(1, H, S, D)
    yt.scaled_dot_product_attention(q, k, v, mask="causal", out=out, backend="math")
    ulp = {torch.float32: 2e-6, torch.bfloat16: 2.0 ** -7}[dt]
    assert ((out.double() - want).abs() <= ulp * float(v.double().abs().max())).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Sq,Skv", [(1, 4100), (3, 5000), (65, 4099)])
def test_sdpa_math_few_queries_many_keys(yt, dev, Sq, Skv, dt):
    """The aligned layouts that take the separate launches (few workgroups, many keys),
    GQA 2:1, against float64. Bound as in test_sdpa_math_one_launch."""
    g = torch.Generator(device=dev).manual_seed(Sq + Skv)
    D = 64
    q = torch.randn(1, 4, Sq, D, device=dev, generator=g).to(dt)
    k = torch.randn(1, 2, Skv, D, device=dev, generator=g).to(dt)
    v = torch.randn(1, 2, Skv, D, device=dev, generator=g).to(dt)
    i, j = torch.arange(Sq, device=dev)[:, None], torch.arange(Skv, device=dev)[None, :]
    drop = torch.rand(Sq, Skv, device=dev, generator=g) < 0.4
    drop[Sq // 2] = True
    bias = torch.randn(Sq, Skv, device=dev, generator=g)
    ulp = {torch.float32: 2e-7, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dt]
    for mask, vis, bs in [(None, None, None), ("causal", j <= i + Skv - Sq, None), (~drop, ~drop, bias)]:
        out = yt.scaled_dot_product_attention(q, k, v, 0.0, mask=mask, bias=bs, backend="math")[0]
        want = _math64(q[0], k[0], v[0], 1.0 / D ** 0.5, vis, bs)
        bound = (1e-5 + ulp) * float(v.double().abs().max()) + 2 * ulp * want.abs()
        assert ((out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("din,dout", [(torch.float32, torch.bfloat16), (torch.float32, torch.float16),
                                      (torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16),
                                      (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("m,n,k", [(5, 7, 3), (130, 200, 72)])
def test_gemm_masked_output_types(yt, dev, m, n, k, din, dout):
    """A C of any type, kept or filled, with alpha / beta, against float64: (k + 2) 2^-24
    sum|a||b| plus the rounding of the result."""
    g = torch.Generator(device=dev).manual_seed(m)
    A = torch.randn(m, k, device=dev, generator=g).to(din)
    B = torch.randn(k, n, device=dev, generator=g).to(din)
    vis = torch.rand(m, n, device=dev, generator=g) < 0.5
    prod, mass = A.double() @ B.double(), A.double().abs() @ B.double().abs()
    ulp = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[dout]
    for alpha, beta, fill in [(1.0, 0.0, -3.0), (1.0, 0.0, None), (0.5, 2.0, 7.0), (0.5, 0.0, None)]:
        C = torch.randn(m, n, device=dev, generator=g).to(dout)
        C0 = C.double()
        yt.gemm_masked(A, B, C, vis, alpha, beta, fill)
        want = alpha * prod + beta * C0
        bound = (k + 2) * 2.0 ** -24 * mass + ulp * want.abs() + 4 * 2.0 ** -23 * C0.abs() + 1e-7
        assert ((C.double() - want).abs() <= bound)[vis].all()
        assert torch.equal(C.double()[~vis], (C0 if fill is None else torch.full_like(C0, fill))[~vis])


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("where", ["a", "b", "a_shifted", "apart_in_one_buffer"])
def test_gemm_masked_output_over_an_input(yt, dev, where, dt):
    """C over A or B (whole, or shifted by some rows) gives the result of a C apart from them:
    with the mask in the product's store, tiles of C would be written while others
    still read A and B. Against float64 as in test_gemm_masked_layouts; kept entries are
    the input's."""
    g = torch.Generator(device=dev).manual_seed(6)
    n = 1024
    buf = (torch.randn(3 * n * n, device=dev, generator=g) * 0.25).to(dt)
    a, b = buf[:n * n].view(n, n), buf[n * n:2 * n * n].view(n, n)
    vis = torch.rand(n, n, device=dev, generator=g) < 0.5
    at = {"a": 0, "b": n * n, "a_shifted": 72 * n, "apart_in_one_buffer": 2 * n * n}[where]
    c = buf[at:at + n * n].view(n, n)
    c0, prod, mass = c.clone(), a.double() @ b.double(), a.double().abs() @ b.double().abs()
    ulp = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -8}[dt]
    yt.gemm_masked(a, b, c, vis)
    assert ((c.double() - prod).abs() <= (n + 2) * 2.0 ** -24 * mass + ulp * prod.abs())[vis].all()
    assert torch.equal(c[~vis], c0[~vis])


@pytest.mark.parametrize("dt,nt,m,n,k", [(torch.bfloat16, False, 3584, 3592, 3072), (torch.float16, True, 3600, 3584, 4104),
                                         (torch.bfloat16, True, 1, 1000, 4096), (torch.bfloat16, True, 16, 1024, 8192),
                                         (torch.bfloat16, False, 1, 1024, 8192), (torch.float32, True, 7, 1000, 1024),
                                         (torch.float32, False, 1, 1024, 1000), (torch.float32, False, 3, 1004, 2048)])
def test_gemm_masked_through_the_workspace(yt, dev, dt, nt, m, n, k):
    """Sizes that run as an fp32 product in the workspace and a blend (256-wide tiles with a
    long k, few rows), with a contiguous and a strided C, each mask kind, kept and filled,
    against float64 as in test_gemm_masked_layouts."""
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    A = torch.randn(m, k, device=dev, generator=g).to(dt)
    B = torch.randn(n, k, device=dev, generator=g).to(dt).t() if nt else torch.randn(k, n, device=dev, generator=g).to(dt)
    prod = A.double() @ B.double().contiguous()
    mass = A.double().abs() @ B.double().abs().contiguous()
    i, j = torch.arange(m, device=dev)[:, None], torch.arange(n, device=dev)[None, :]
    bytes_ = torch.rand(m, n, device=dev, generator=g) < 0.5
    ulp = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[dt]
    for mask, vis in [("causal", j <= i + n - m), (("diag", 5), j <= i + 5), (bytes_, bytes_)]:
        for alpha, beta, fill, step in [(1.0, 0.0, -3.0, 1), (0.5, 2.0, None, 1), (1.0, 0.0, None, 2)]:
            C = torch.randn(m, step * n, device=dev, generator=g).to(dt)[:, ::step]
            C0 = C.double()
            yt.gemm_masked(A, B, C, mask, alpha, beta, fill)
            want = alpha * prod + beta * C0
            bound = (k + 2) * 2.0 ** -24 * mass + ulp * want.abs() + 4 * 2.0 ** -23 * C0.abs() + 1e-7
            ok = (C.double() - want).abs() <= bound
            assert ok[vis.expand(m, n)].all(), (mask if isinstance(mask, (str, tuple)) else "bytes", alpha, fill)
            hid = (~vis).expand(m, n)
            assert torch.equal(C.double()[hid], (C0 if fill is None else torch.full_like(C0, fill))[hid])
