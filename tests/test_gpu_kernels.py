"""Operator-level parity of the HIP kernels (GPU).

Each kernel is called through the C ABI (``rwkv_tl_amd.kernels``) and compared
with the CPU oracle or a plain fp32 torch computation of the same op on the
same seeded inputs:

* wkv7 (standalone DPLR, config C2 and edge shapes) vs ``oracle.wkv7_scan``:
  y within 1 fp16 ulp-ish (rtol 2e-3, atol 2e-3), fp32 state within 1e-5
  relative (Frobenius) -- the kernel and the oracle both accumulate in fp32.
* GEMV / GEMM (every epilogue) vs fp32 torch on the same fp16 operands.
* LayerNorm vs ``F.layer_norm``; token-shift lerps vs the closed form with the
  reference's test tolerance (test/test_kernels.py:17-43: fp16, C=768, seeds
  42..49, 0.01).
* The time-mix stage operators (single gates, fused gates, packed LoRA first
  step, L2 norm, GroupNorm + bonus) vs the oracle's operator restatements on
  the same fp16 inputs: f16 outputs within rtol 4e-3, atol 4e-3 (one or two
  fp16 ulps at these magnitudes; both sides compute in fp32).
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from oracle import rwkv7_ref as R
from rwkv_tl_amd import kernels as K

pytestmark = pytest.mark.gpu


def _c2_inputs(B, H, T, seed=0, w_f32=True):
    """Config C2 recipe: r,k,v ~ N(0,1) fp16; w = exp(-exp(x)), x ~ N(-0.5, 0.5);
    a = -kappa, b = kappa * alpha with kappa the per-head L2-normalised k and
    alpha = sigmoid(N(0,1)); S0 ~ N(0, 0.1^2) fp32."""
    g = torch.Generator().manual_seed(seed)
    shp = (B, T, H, 64)
    r = torch.randn(shp, generator=g).half()
    k = torch.randn(shp, generator=g).half()
    v = torch.randn(shp, generator=g).half()
    w = torch.exp(-torch.exp(torch.randn(shp, generator=g) * 0.5 - 0.5))
    kap = F.normalize(k.float(), dim=-1)
    alpha = torch.sigmoid(torch.randn(shp, generator=g))
    a = (-kap).half()
    b = (kap * alpha).half()
    S0 = torch.randn(B, H, 64, 64, generator=g) * 0.1
    return S0, r, (w if w_f32 else w.half()), k, v, a, b


def _rel(x, y):
    return float((x.double() - y.double()).norm() / y.double().norm().clamp_min(1e-30))


@pytest.mark.parametrize("chunked", [False, True], ids=["serial", "chunked"])
@pytest.mark.parametrize(
    "B,H,T,w_f32",
    [(8, 16, 128, True), (1, 1, 1, True), (2, 3, 17, False), (1, 4, 33, True), (3, 2, 64, False),
     (4, 32, 40, False)],
)
def test_wkv7_matches_oracle(B, H, T, w_f32, chunked, cuda):
    """Both algorithms (rwkv7_wkv7, rwkv7_wkv7_chunked) against the serial
    fp32 oracle: the state within 1e-5 relative, y (f16) within 2e-3. T = 1,
    17, 33 and 40 leave the chunked form a partial last chunk; 8 x 16 and
    4 x 32 heads fill every CU with chain workgroups."""
    print(f"wkv7 B={B} H={H} T={T} w_f32={w_f32} chunked={chunked}", flush=True)
    S0, r, w, k, v, a, b = _c2_inputs(B, H, T, seed=B * 100 + T, w_f32=w_f32)
    y_ref, S_ref = R.wkv7_scan(S0, r, w, k, v, a, b)
    S = S0.clone().to(cuda)
    y = K.wkv7(S, *(t.to(cuda) for t in (r, w, k, v, a, b)), chunked=chunked)
    torch.cuda.synchronize()
    assert _rel(S.cpu(), S_ref) < 1e-5
    torch.testing.assert_close(y.cpu().float(), y_ref.float(), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("w_low", [1e-3, 0.0], ids=["tiny", "zero"])
def test_wkv7_chunked_strong_decay(w_low, cuda):
    """Decays whose 16-token products leave [1e-30, 1e30] (tiny or zero w on
    some channels) take the chunked kernel's direct-product branch for those
    chunks; results still match the oracle, and no value is lost to an
    overflow of the reciprocal products."""
    B, H, T = 2, 3, 48
    S0, r, w, k, v, a, b = _c2_inputs(B, H, T, seed=5, w_f32=True)
    w = w.clone()
    w[0, 16:32, :, :8] = w_low  # chunk 1 of sequence 0: slow branch; the rest fast
    w[1, :, 1, 60:] = w_low
    y_ref, S_ref = R.wkv7_scan(S0, r, w, k, v, a, b)
    S = S0.clone().to(cuda)
    y = K.wkv7(S, *(t.to(cuda) for t in (r, w, k, v, a, b)), chunked=True)
    torch.cuda.synchronize()
    assert torch.isfinite(S).all() and torch.isfinite(y.float()).all()
    assert _rel(S.cpu(), S_ref) < 1e-5
    torch.testing.assert_close(y.cpu().float(), y_ref.float(), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("H", [3, 64])
@pytest.mark.parametrize("chunked", [False, True], ids=["serial", "chunked"])
def test_wkv7_closed_forms(chunked, H, cuda):
    """Two closed forms of the recurrence (both algorithms, three 16-token
    chunks): with w = 1 and a = b = 0 the state accumulates sum_t v_t k_t^T
    and y_t = S_t r_t; with k = v = 0 and a = b = 0 each key column of the
    state decays by the product of its w. H = 64 (B H = 128) fills every CU
    with chain workgroups."""
    B, T, N = 2, 48, 64
    g = torch.Generator().manual_seed(12)
    S0 = torch.randn(B, H, N, N, generator=g, dtype=torch.float64) * 0.1
    r, k, v = (torch.randn(B, T, H, N, generator=g).half() for _ in range(3))
    zero = torch.zeros(B, T, H, N).half()
    # accumulation: S_t = S_0 + sum_{s<=t} v_s k_s^T
    S = S0.float().to(cuda)
    y = K.wkv7(S, r.to(cuda), torch.ones(B, T, H, N).to(cuda), k.to(cuda), v.to(cuda), zero.to(cuda),
               zero.to(cuda), chunked=chunked)
    vk = torch.einsum("bthi,bthj->bthij", v.double(), k.double()).cumsum(1)  # [B, T, H, N, N]
    St = S0.unsqueeze(1) + vk
    y_ref = torch.einsum("bthij,bthj->bthi", St, r.double())
    torch.cuda.synchronize()
    assert _rel(S.cpu(), St[:, -1]) < 1e-5
    torch.testing.assert_close(y.cpu().double(), y_ref, rtol=2e-3, atol=2e-2)
    # decay: S_T = S_0 diag(prod_t w_t)
    w = torch.exp(-torch.exp(torch.randn(B, T, H, N, generator=g) * 0.5 - 0.5))
    S = S0.float().to(cuda)
    K.wkv7(S, r.to(cuda), w.to(cuda), zero.to(cuda), zero.to(cuda), zero.to(cuda), zero.to(cuda), chunked=chunked)
    torch.cuda.synchronize()
    want = S0 * w.double().prod(1).unsqueeze(2)  # column j scaled by prod_t w_t[j]
    assert _rel(S.cpu(), want) < 1e-5


@pytest.mark.parametrize("B,H", [(2, 2), (4, 32)])
def test_wkv7_chunked_long_sequence_agrees_with_serial(B, H, cuda):
    """T = 1024 (the C5 prefill length) in bfloat16: the chunked and serial
    algorithms agree on the final state to 1e-4 relative and on y to bf16
    rounding; 4 x 32 is the C5 shape."""
    T = 1024
    S0, r, w, k, v, a, b = _c2_inputs(B, H, T, seed=9, w_f32=True)
    ins = [t.to(cuda) for t in (r, w, k, v, a, b)]
    ins = [t.bfloat16() if t.dtype == torch.float16 else t for t in ins]
    outs = []
    for chunked in (False, True):
        S = S0.clone().to(cuda)
        y = K.wkv7(S, *ins, chunked=chunked)
        outs.append((S.cpu(), y.float().cpu()))
    torch.cuda.synchronize()
    assert _rel(outs[1][0], outs[0][0]) < 1e-4
    torch.testing.assert_close(outs[1][1], outs[0][1], rtol=2e-2, atol=2e-2)


def test_fused_dplr_step_and_sequence_api(cuda):
    S0, r, w, k, v, a, b = _c2_inputs(1, 4, 5, seed=7, w_f32=False)
    S = S0[0].clone().to(cuda)
    ys = []
    for t in range(5):
        y, S = K.fused_dplr(S, *(x[0, t].to(cuda) for x in (r, w, k, v, a, b)))
        ys.append(y)
    S2 = S0[0].clone().to(cuda)
    y2, S2 = K.fused_dplr_T(S2, *(x[0].to(cuda) for x in (r, w, k, v, a, b)))
    torch.testing.assert_close(torch.stack(ys), y2, rtol=0, atol=0)
    torch.testing.assert_close(S, S2, rtol=0, atol=0)


def test_wkv7_rejects_bad_shapes(cuda):
    S0, r, w, k, v, a, b = _c2_inputs(1, 2, 3)
    S = S0.to(cuda)
    with pytest.raises(ValueError):
        K.wkv7(S, r.to(cuda), w.to(cuda), k.to(cuda)[:, :2], v.to(cuda), a.to(cuda), b.to(cuda))
    with pytest.raises(ValueError):
        K.wkv7(S.double(), *(t.to(cuda) for t in (r, w, k, v, a, b)))


@pytest.mark.parametrize("N,Kd", [(8, 256), (1000, 768), (3360, 1024), (1024, 4096), (4096, 1024), (2048, 8192)])
def test_gemv_matches_fp32(N, Kd, cuda):
    g = torch.Generator().manual_seed(N + Kd)
    W = (torch.randn(N, Kd, generator=g) * 0.02).half()
    x = torch.randn(Kd, generator=g)
    y = K.gemv(x.to(cuda), W.to(cuda)).cpu()
    ref = W.float() @ x
    torch.testing.assert_close(y, ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize(
    "M,N,Kd",
    [(1, 64, 256), (5, 100, 40), (16, 1024, 1024), (33, 72, 16), (128, 4096, 1024), (200, 1024, 4096), (7, 65536, 256),
     # mid M on the 32/64-row tiled kernels
     (512, 1024, 1024), (600, 300, 128), (1030, 520, 64),
     # large-M path: 256 x 256 tiles (also ragged), 128 x 128 tiles (also ragged)
     (2048, 8192, 1024), (4000, 4000, 64), (4096, 2048, 2048), (2100, 3900, 128)],
)
@pytest.mark.parametrize("epi", ["f32", "f16", "relu2", "add"])
def test_gemm_matches_fp32(M, N, Kd, epi, cuda):
    g = torch.Generator().manual_seed(M * 7 + N + Kd)
    A = torch.randn(M, Kd, generator=g).half()
    W = (torch.randn(N, Kd, generator=g) * 0.05).half()
    ref = A.float() @ W.float().T
    if epi == "add":
        base = torch.randn(M, N, generator=g)
        out = K.gemm(A.to(cuda), W.to(cuda), "add", out=base.clone().to(cuda)).cpu()
        torch.testing.assert_close(out, base + ref, rtol=1e-4, atol=1e-4)
        return
    out = K.gemm(A.to(cuda), W.to(cuda), epi).cpu().float()
    if epi == "relu2":
        ref = ref.clamp_min(0) ** 2
    if epi == "f32":
        torch.testing.assert_close(out, ref, rtol=1e-4, atol=1e-4)
    else:
        torch.testing.assert_close(out, ref.half().float(), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("M,N,Kd", [(2048, 8192, 1024), (4096, 2048, 2048), (2100, 3900, 128)])
@pytest.mark.parametrize("epi", ["f32", "f16", "relu2", "add"])
def test_gemm_bf16_large_m_matches_fp32(M, N, Kd, epi, cuda):
    """bfloat16 operands on the large-M path (hipBLASLt for the plain
    epilogues, the large-M kernel for relu2): the products of bf16 values are
    exact in fp32, so f32 outputs must match the fp32 product to fp32
    accumulation accuracy and 16-bit outputs its bfloat16 rounding."""
    g = torch.Generator().manual_seed(M * 5 + N + Kd)
    A = torch.randn(M, Kd, generator=g).bfloat16()
    W = (torch.randn(N, Kd, generator=g) * 0.05).bfloat16()
    ref = A.float() @ W.float().T
    if epi == "add":
        base = torch.randn(M, N, generator=g)
        out = K.gemm(A.to(cuda), W.to(cuda), "add", out=base.clone().to(cuda)).cpu()
        torch.testing.assert_close(out, base + ref, rtol=1e-4, atol=1e-4)
        return
    out = K.gemm(A.to(cuda), W.to(cuda), epi).cpu().float()
    if epi == "relu2":
        ref = ref.clamp_min(0) ** 2
    if epi == "f32":
        torch.testing.assert_close(out, ref, rtol=1e-4, atol=1e-4)
    else:
        torch.testing.assert_close(out, ref.bfloat16().float(), rtol=8e-3, atol=8e-3)


@pytest.mark.parametrize("M,N,Kd", [(2048, 8192, 1024), (2100, 3900, 128)])
def test_gemm_large_m_relu2_squares_the_half_product(M, N, Kd, cuda):
    """On the large-M path half relu2 runs as hipBLASLt's half product
    followed by an in-place pass (eight values per access where N allows, one
    at a time otherwise: N = 3900): its output must equal, bit for bit,
    relu(p)^2 rounded to half, where p is the same shape's "f16" output (the
    same algorithm: the plan depends on the shape only) -- the rounding of the
    reference's fp16 path, relu(x @ W^T) ** 2 on a half product."""
    g = torch.Generator().manual_seed(M * 3 + N + Kd)
    A = torch.randn(M, Kd, generator=g).half().to(cuda)
    W = (torch.randn(N, Kd, generator=g) * 0.05).half().to(cuda)
    p = K.gemm(A, W, "f16")
    y = K.gemm(A, W, "relu2")
    want = (p.float().clamp_min(0) ** 2).half()
    assert torch.equal(y, want), f"{(y.float() - want.float()).abs().max().item():.3e}"


@pytest.mark.parametrize("epi", ["relu2", "f32"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_gemm_large_m_first_seen_under_capture(epi, dt, cuda):
    """A large-M shape seen first inside a graph capture runs this library's
    own large-M kernel (no hipBLASLt plan is built while the stream captures);
    the same call made eagerly afterwards builds the plan and runs hipBLASLt
    (bf16 relu2 stays on the own kernel). Every replay (each after eager work
    that overwrites its output) and the eager call must match the fp32
    product: f32 to fp32 accumulation accuracy, relu2 to the 16-bit format's
    rounding. The shape is this test's own (N differs per case), so no
    earlier call in the process has built its plan."""
    M, Kd = 2304, 256
    N = 4352 + (64 if dt == torch.bfloat16 else 0) + (128 if epi == "f32" else 0)
    g = torch.Generator().manual_seed(N)
    A = torch.randn(M, Kd, generator=g).to(dt)
    W = (torch.randn(N, Kd, generator=g) * 0.05).to(dt)
    ref = A.float() @ W.float().T
    if epi == "relu2":
        ref = ref.clamp_min(0) ** 2
    A, W = A.to(cuda), W.to(cuda)
    K.gemm(A[:8], W[:64], "f32")  # library loaded, device queried, outside the capture
    torch.cuda.synchronize()

    def check(out, what):
        out = out.cpu().float()
        if epi == "f32":
            torch.testing.assert_close(out, ref, rtol=1e-4, atol=1e-4, msg=what)
        elif dt == torch.float16:
            torch.testing.assert_close(out, ref.half().float(), rtol=2e-3, atol=2e-3, msg=what)
        else:
            torch.testing.assert_close(out, ref.bfloat16().float(), rtol=8e-3, atol=8e-3, msg=what)

    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = K.gemm(A, W, epi)
    check(K.gemm(A, W, epi), "eager after the capture")
    for i in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        check(out, f"replay {i}")


@pytest.mark.parametrize(
    "M,N,Kd",
    [(1, 64, 256), (5, 100, 40), (8, 300, 1024), (12, 1024, 4096), (16, 1024, 1024), (24, 4096, 1024),
     (33, 72, 16), (128, 4096, 1024), (128, 1024, 4096),
     (200, 1024, 4096), (7, 65536, 256), (512, 1024, 1024), (600, 300, 128), (1030, 520, 64), (2048, 1024, 256)],
)
@pytest.mark.parametrize("epi", ["f32", "add", "relu2_f32", "tanh_f32", "sigmoid_f32", "f16"])
@pytest.mark.parametrize("wdt", [torch.float16, torch.bfloat16])
def test_gemm_f32_activations_match_fp32(M, N, Kd, epi, wdt, cuda):
    """f32 A (the model's batched and prefill GEMM operands): the kernels split
    each activation into its 16-bit part and the 16-bit remainder and multiply
    both by the weight fragment, so the product must equal the float64 product
    of the f32 activations and the 16-bit weights to fp32 accuracy: within
    tol (1 + |x|) of the pre-activation x, carried through the activation by
    its derivative, with tol = 1e-6 sqrt(K) for half (the fp32 accumulation
    over K: hi + lo hold 22 significant bits) and 4e-6 sqrt(K) for bfloat16
    (16 bits). The same bar is shown to fail for A rounded to the 16-bit
    format (an error near 2^-12 sqrt(K) |w| per output), so it sees the split."""
    g = torch.Generator().manual_seed(M * 11 + N + Kd)
    A = torch.randn(M, Kd, generator=g)
    W = (torch.randn(N, Kd, generator=g) * 0.05).to(wdt)
    x = A.double() @ W.double().T
    tol = (1e-6 if wdt == torch.float16 else 4e-6) * Kd**0.5
    dx = tol * (1.0 + x.abs())  # allowed error of the pre-activation
    if epi == "add":
        base = torch.randn(M, N, generator=g)
        out = K.gemm(A.to(cuda), W.to(cuda), "add", out=base.clone().to(cuda)).cpu().double() - base.double()
        want, bar = x, dx + 1e-6 * base.double().abs()
    elif epi == "f16":
        # the 16-bit store rounds the product; it must be the rounding of x
        out = K.gemm(A.to(cuda), W.to(cuda), epi).cpu().double()
        want, bar = x.to(wdt).double(), x.abs() * (2.0**-10 if wdt == torch.float16 else 2.0**-7) + dx
    else:
        out = K.gemm(A.to(cuda), W.to(cuda), epi).cpu().double()
        if epi == "relu2_f32":
            want, bar = x.clamp_min(0) ** 2, 2.0 * x.abs() * dx + dx**2
        elif epi == "tanh_f32":
            want, bar = torch.tanh(x), dx
        elif epi == "sigmoid_f32":
            want, bar = torch.sigmoid(x), dx
        else:
            want, bar = x, dx
    d = (out - want).abs()
    assert bool((d <= bar).all()), f"{int((d > bar).sum())} off, max |d| {float(d.max()):.3e}"
    if epi == "f32" and M * N * Kd >= 1 << 20:
        rounded = A.to(wdt).double() @ W.double().T
        assert bool(((rounded - x).abs() > dx).any()), "the bar does not see 16-bit activations"


@pytest.mark.slow
def test_gemm_large_m_beyond_2gib_of_a(cuda):
    """The large-M GEMM reads its operands through 32-bit buffer offsets, so an
    A of 2 GiB or more runs as row blocks of whole 256-row tiles below 2^31
    bytes each (lda 8192: 130816 rows per block). A [131392, 8192] f16 is
    2.15 GB; rows on both sides of the block boundary, the first rows and the
    last rows must equal the fp32 product, in both the f32 and add epilogues."""
    M, N, Kd = 131392, 256, 8192
    boundary = (2**31 - 1) // (2 * Kd) // 256 * 256
    assert boundary == 130816
    print(f"gemm M={M} N={N} K={Kd}: A {M * Kd * 2 / 2**30:.2f} GiB, block boundary row {boundary}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(3)
    A = torch.randn(M, Kd, generator=g, device=cuda, dtype=torch.float16)
    W = (torch.randn(N, Kd, generator=g, device=cuda) * 0.05).half()
    rows = torch.cat([torch.arange(0, 40), torch.arange(boundary - 300, boundary + 300), torch.arange(M - 40, M)])
    ref = (A[rows.to(cuda)].float().cpu() @ W.float().cpu().T)
    out = K.gemm(A, W, "f32")
    torch.testing.assert_close(out[rows.to(cuda)].cpu(), ref, rtol=1e-4, atol=1e-4)
    base = torch.randn(M, N, generator=g, device=cuda)
    want = base[rows.to(cuda)].cpu() + ref
    K.gemm(A, W, "add", out=base)
    torch.testing.assert_close(base[rows.to(cuda)].cpu(), want, rtol=1e-4, atol=1e-4)
    del A, base, out
    torch.cuda.empty_cache()


def test_fused_rkv_gemm_matches_reference_layout(cuda):
    g = torch.Generator().manual_seed(5)
    T, C = 9, 256
    xs = [torch.randn(T, C, generator=g).half() for _ in range(3)]
    Wb = (torch.randn(3, C, C, generator=g) * 0.05).half()  # [3, in, out] as in weight.py:98-105
    out = K.fused_rkv_gemm(*(x.to(cuda) for x in xs), Wb.to(cuda)).cpu().float()
    ref = torch.stack([xs[i].float() @ Wb[i].float() for i in range(3)])
    torch.testing.assert_close(out, ref, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("C", [256, 768, 1024, 4096])
def test_layernorm_matches_torch(C, cuda):
    g = torch.Generator().manual_seed(C)
    x = torch.randn(5, C, generator=g) * 3 + 1
    w = torch.randn(C, generator=g)
    b = torch.randn(C, generator=g)
    y = K.layer_norm(x.to(cuda), w.to(cuda), b.to(cuda)).cpu()
    torch.testing.assert_close(y, F.layer_norm(x, (C,), w, b), rtol=1e-5, atol=1e-5)
    y16 = K.layer_norm(x.half().to(cuda), w.to(cuda), b.to(cuda)).cpu()
    torch.testing.assert_close(y16, F.layer_norm(x.half().float(), (C,), w, b), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("seed", [42 + i for i in range(8)])
def test_fused_lerp6_exact(seed, cuda):
    """Reference test/test_kernels.py:17-43 (fp16, C=768, tolerance 0.01)."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(768, generator=g).half()
    prev = torch.randn(768, generator=g).half()
    ws = [torch.randn(768, generator=g).half() for _ in range(6)]
    got = K.fused_lerp6(x.to(cuda), prev.to(cuda), *(w.to(cuda) for w in ws))
    for w, o in zip(ws, got):
        ref = x + w * (prev - x)
        assert (ref.float() - o.cpu().float()).abs().max().item() <= 0.01


def test_lerp_copy_variants_update_state_after_read(cuda):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(1024, generator=g).half().to(cuda)
    prev = torch.randn(1024, generator=g).half().to(cuda)
    mu = torch.rand(1024, generator=g).half().to(cuda)
    prev0 = prev.clone()
    # x_copy aliases prev, as in the model (lerp.py:190-198)
    out = K.fused_lerp1_copy(x, prev, mu, prev)
    ref = x.float() + mu.float() * (prev0.float() - x.float())
    assert (out.float() - ref).abs().max().item() <= 0.01
    assert torch.equal(prev, x)
    buf = torch.zeros_like(x)
    outs = K.fused_lerp6_copy(x, prev0, *([mu] * 6), buf)
    assert len(outs) == 6 and torch.equal(buf, x)


# --------------------------------------------------------------------------
# time-mix stage operators
# --------------------------------------------------------------------------

OP_TOL = dict(rtol=4e-3, atol=4e-3)


def _h(g, *shape, scale=1.0, shift=0.0):
    return (torch.randn(*shape, generator=g) * scale + shift).half()


@pytest.mark.parametrize("C", [1, 768, 1024, 4099])
def test_single_gates_match_oracle(C, cuda):
    g = torch.Generator().manual_seed(C)
    x, w0, v, vf, v0, v12, a0, ax, k, kk, ka = (_h(g, C) for _ in range(11))
    dev = lambda *ts: [t.to(cuda) for t in ts]  # noqa: E731
    torch.testing.assert_close(K.fused_w_gate(*dev(x, w0)).cpu().float(), R.w_gate(x, w0), **OP_TOL)
    torch.testing.assert_close(K.fused_v_gate(*dev(v, vf, v0, v12)).cpu().float(), R.v_gate(v, vf, v0, v12), **OP_TOL)
    got = K.fused_a_kk_k(*dev(a0, ax, k, kk, ka))
    for gg, ww in zip(got, R.a_kk_k(a0, ax, k, kk, ka)):
        torch.testing.assert_close(gg.cpu().float(), ww, **OP_TOL)


@pytest.mark.parametrize("C,ranks", [(1024, (32, 64, 64, 128)), (768, (16, 32, 32, 64)), (256, (8, 24, 40, 72))])
def test_fused_gates_match_oracle(C, ranks, cuda):
    g = torch.Generator().manual_seed(C + sum(ranks))
    rv, rw, ra, rg = ranks
    vr, wr, ar, gr = (_h(g, r) for r in ranks)
    mats = [_h(g, C, r, scale=0.1) for r in ranks]
    vecs = [_h(g, C) for _ in range(8)]  # v, v_first, k, v0, w0, a0, k_k, k_a
    args = (vr, wr, ar, gr, *vecs[:3], *mats, *vecs[3:])
    got = K.fused_gates(*(t.to(cuda) for t in args))
    want = R.gates(*args)
    for name, gg, ww in zip(("v", "w", "a", "kk", "k", "g"), got, want):
        torch.testing.assert_close(gg.cpu().float(), ww, **OP_TOL, msg=name)


@pytest.mark.parametrize("C,ranks", [(1024, (32, 64, 64, 128)), (2048, (64, 64, 96, 256)), (256, (8, 24, 40, 72))])
def test_fused_rank_gemv_matches_oracle(C, ranks, cuda):
    g = torch.Generator().manual_seed(C)
    xs = [_h(g, C) for _ in range(4)]
    packed = _h(g, sum(ranks), C, scale=0.05)
    got = K.fused_rank_gemv(*(t.to(cuda) for t in xs), packed.to(cuda), *ranks)
    torch.testing.assert_close(got.cpu().float(), R.rank_gemv(*xs, packed, *ranks), **OP_TOL)


@pytest.mark.parametrize("H", [1, 12, 16, 33])
def test_l2norm_and_gn_rkrk_match_oracle(H, cuda):
    g = torch.Generator().manual_seed(H)
    kk, a = _h(g, H, 64), torch.rand(H, 64, generator=g).half()
    kk[0] = 0  # the zero head: clamped denominator, outputs stay zero
    kn, b = K.fused_l2norm_neg_kk_a(kk.to(cuda), a.to(cuda))
    wkn, wb = R.l2norm_neg_kk_a(kk, a)
    torch.testing.assert_close(kn.cpu().float(), wkn, **OP_TOL)
    torch.testing.assert_close(b.cpu().float(), wb, **OP_TOL)
    y, r, k, v, rk = (_h(g, H, 64) for _ in range(5))
    lw, lb = _h(g, H * 64, scale=0.2, shift=1.0), _h(g, H * 64, scale=0.2)
    got = K.fused_gn_rkrk(*(t.to(cuda) for t in (y, r, k, v, rk, lw, lb)))
    torch.testing.assert_close(got.cpu().float(), R.gn_rkrk(y, r, k, v, rk, lw, lb), rtol=1e-2, atol=1e-2)


def test_stage_operators_reject_bad_shapes(cuda):
    h = lambda *s: torch.zeros(*s, dtype=torch.float16, device=cuda)  # noqa: E731
    with pytest.raises(ValueError):
        K.fused_w_gate(h(8), h(9))
    with pytest.raises(ValueError):
        K.fused_l2norm_neg_kk_a(h(2, 32), h(2, 32))
    with pytest.raises(ValueError):
        K.fused_rank_gemv(h(64), h(64), h(64), h(64), h(10, 64), 2, 2, 2, 2)
    with pytest.raises(ValueError):
        K.fused_w_gate(h(8).float(), h(8))


def _dplr_inputs(B, T, H, seed):
    """Inputs shaped like a real step: w = exp(-exp(x)) in (0, 1), a the
    L2-normalised key per head, b = -a * sigmoid(.), state ~ N(0, 0.1)."""
    g = torch.Generator().manual_seed(seed)
    S = torch.randn(B, H, 64, 64, generator=g) * 0.1
    r, k, v = (torch.randn(B, T, H, 64, generator=g) * 0.5 for _ in range(3))
    w = torch.exp(-torch.exp(torch.randn(B, T, H, 64, generator=g) * 0.5 - 0.5))
    kh = torch.nn.functional.normalize(torch.randn(B, T, H, 64, generator=g), dim=-1)
    a = kh
    b = -kh * torch.sigmoid(torch.randn(B, T, H, 64, generator=g))
    return S, r, w, k, v, a, b


def _rel(x, y):
    return float((x.double() - y.double()).norm() / y.double().norm().clamp_min(1e-30))


@pytest.mark.parametrize("B,T,H,with_gS", [(1, 1, 1, True), (2, 20, 3, True), (1, 37, 2, False), (2, 130, 1, True)])
def test_wkv7_backward_matches_oracle(B, T, H, with_gS, cuda):
    """Reverse-time adjoint scan (rwkv7_wkv7_backward) against the oracle's
    autograd gradients of the serial fp32 scan; every gradient within 2e-4
    relative (Frobenius) and elementwise within 2e-4 of its scale. The forward
    with history (rwkv7_wkv7_f32) must match the oracle's y and final state."""
    S, r, w, k, v, a, b = _dplr_inputs(B, T, H, seed=100 * T + H)
    g = torch.Generator().manual_seed(7)
    gy = torch.randn(B, T, H, 64, generator=g)
    gS = torch.randn(B, H, 64, 64, generator=g) if with_gS else None
    ref = R.wkv7_scan_grads(S, r, w, k, v, a, b, gy, gS)
    y_ref, S_ref = R.wkv7_scan(S, r, w, k, v, a, b)

    d = [x.to(cuda) for x in (S, r, w, k, v, a, b)]
    Sg = d[0].clone()
    hist = torch.empty(B, H, T, 64, 64, device=cuda)
    y = K.wkv7_f32(Sg, *d[1:], hist=hist)
    assert _rel(y.cpu(), y_ref) < 1e-5 and _rel(Sg.cpu(), S_ref) < 1e-5
    assert torch.allclose(hist[:, :, 0].cpu(), S)  # the state entering step 0 is S0
    got = K.wkv7_backward(hist, Sg, *d[1:], gy.to(cuda), None if gS is None else gS.to(cuda))
    for name, x, xr in zip(("S0", "r", "w", "k", "v", "a", "b"), got, ref):
        x = x.cpu()
        assert _rel(x, xr) < 2e-4, f"grad {name}: rel {_rel(x, xr):.2e}"
        assert torch.allclose(x, xr, rtol=0, atol=2e-4 * float(xr.abs().max())), f"grad {name}"


def test_dplr_seq_operator_autograd(cuda):
    """torch.ops.rwkv_tl.fused_dplr_seq with torch.library.register_autograd:
    loss.backward() through the HIP forward and backward gives the oracle's
    gradients, unbatched ([H,64,64] / [T,H,64]) as the reference's fused_dplr_T
    shapes; S itself is left unchanged."""
    import rwkv_tl_amd.operators  # noqa: F401  (registers the operators)

    S, r, w, k, v, a, b = _dplr_inputs(1, 24, 2, seed=5)
    g = torch.Generator().manual_seed(9)
    gy = torch.randn(24, 2, 64, generator=g)
    gS = torch.randn(2, 64, 64, generator=g)
    xs = [t[0].to(cuda).requires_grad_(True) for t in (S, r, w, k, v, a, b)]
    S_before = xs[0].detach().clone()
    y, S_T = torch.ops.rwkv_tl.fused_dplr_seq(*xs)
    ((y * gy.to(cuda)).sum() + (S_T * gS.to(cuda)).sum()).backward()
    assert torch.equal(xs[0].detach(), S_before)
    ref = R.wkv7_scan_grads(S, r, w, k, v, a, b, gy.unsqueeze(0), gS.unsqueeze(0))
    for name, x, xr in zip(("S0", "r", "w", "k", "v", "a", "b"), xs, ref):
        assert _rel(x.grad.cpu(), xr[0]) < 2e-4, f"grad {name}"


@pytest.mark.parametrize("B,T,H,with_gS,decay", [
    (1, 1, 1, True, "plain"), (1, 15, 2, False, "plain"), (2, 16, 1, True, "plain"), (1, 17, 3, True, "plain"),
    (1, 24, 1, True, "plain"), (2, 129, 2, True, "plain"), (1, 40, 2, True, "strong"), (1, 33, 1, False, "zero"),
])
def test_dplr_seq_gradient_matches_oracle(B, T, H, with_gS, decay, cuda):
    """dplr_seq_forward / dplr_seq_backward (chunked scans of the state and of
    its adjoint, then every 16-token chunk at once) against the oracle's
    autograd gradients in fp32, around the chunk (16) and half-chunk (8)
    edges, for two workgroup sizes of the chains, and with decays whose
    products leave the range the scaled form is used in (strong: w^40, products
    below 1e-30 in a chunk; zero: some w = 0). Both sides sum the same fp32
    terms in another order; roundings mostly cancel, and no bound short of the
    worst case (T + 64 ulps, amplified by the recurrence) is derived: the errors
    measured are at most 2.6e-7, and 1e-5 is asserted. (The forward is chunked
    from 128 or 144 tokens only: the strong and zero decays reach its chunked
    form in test_chunked_scans_are_as_exact_as_the_serial_scan.)"""
    S, r, w, k, v, a, b = _dplr_inputs(B, T, H, seed=31 * T + H)
    g = torch.Generator().manual_seed(11)
    if decay == "strong":
        w = w**40
    elif decay == "zero":
        w = torch.where(torch.rand(w.shape, generator=g) < 0.05, torch.zeros_like(w), w)
    gy = torch.randn(B, T, H, 64, generator=g)
    gS = torch.randn(B, H, 64, 64, generator=g) if with_gS else None
    y_ref, S_ref = R.wkv7_scan(S, r, w, k, v, a, b)
    ref = R.wkv7_scan_grads(S, r, w, k, v, a, b, gy, gS)
    d = [x.to(cuda) for x in (S, r, w, k, v, a, b)]
    y, S_T = K.dplr_seq_forward(*d)
    assert _rel(y.cpu(), y_ref) < 1e-5 and _rel(S_T.cpu(), S_ref) < 1e-5
    got = K.dplr_seq_backward(*d, gy.to(cuda), None if gS is None else gS.to(cuda))
    assert torch.equal(d[0].cpu(), S)
    for name, x, xr in zip(("S0", "r", "w", "k", "v", "a", "b"), got, ref):
        assert _rel(x.cpu(), xr) < 1e-5, f"grad {name}: rel {_rel(x.cpu(), xr):.2e}"


def test_dplr_seq_gradient_many_heads_matches_history_backward(cuda):
    """A grid of more heads than CUs (two value quarters per chain workgroup)
    against the history-based backward (rwkv7_wkv7_backward) on the same
    device; both fp32, measured 1.7e-7 apart, 1e-5 as above."""
    d = [x.to(cuda) for x in _dplr_inputs(3, 50, 24, seed=77)]
    gy = torch.randn(3, 50, 24, 64, device=cuda)
    S1 = d[0].clone()
    hist = torch.empty(3, 24, 50, 64, 64, device=cuda)
    K.wkv7_f32(S1, *d[1:], hist=hist)
    want = K.wkv7_backward(hist, S1, *d[1:], gy, None)
    for x, xr in zip(K.dplr_seq_backward(*d, gy, None), want):
        assert _rel(x, xr) < 1e-5


def _grads64(ins, gy, gS):
    """y, S_T and the seven gradients of the recurrence, step by step in 64 bits."""
    S, r, w, k, v, a, b = xs = [x.double().requires_grad_(True) for x in ins]
    ys = []
    for t in range(r.shape[1]):
        sa = torch.matmul(S, a[:, t].unsqueeze(-1))
        S = S * w[:, t].unsqueeze(-2) + sa * b[:, t].unsqueeze(-2) + v[:, t].unsqueeze(-1) * k[:, t].unsqueeze(-2)
        ys.append(torch.matmul(S, r[:, t].unsqueeze(-1)).squeeze(-1))
    y = torch.stack(ys, dim=1)
    return [y.detach(), S.detach(), *torch.autograd.grad((y, S), xs, (gy.double(), gS.double()))]


@pytest.mark.parametrize("decay", ["plain", "strong", "zero"])
def test_chunked_scans_are_as_exact_as_the_serial_scan(decay, cuda):
    """Against 64 bits, the chunked forward and gradient may be no further off
    than the serial scan and the history backward, whose every step rounds: the
    same error to the 5 % by which the rounding of 0.2 million values varies
    between inputs (strong: products of w below 1e-30, zero: some w = 0, the
    direct form)."""
    B, T, H = 2, 160, 10
    ins = [x.to(cuda) for x in _dplr_inputs(B, T, H, seed=3)]
    if decay == "strong":
        ins[2] = ins[2] ** 12
    elif decay == "zero":
        ins[2] = ins[2] * (torch.rand(ins[2].shape, generator=torch.Generator().manual_seed(5)) >= 0.05).to(cuda)
    g = torch.Generator().manual_seed(4)
    gy = torch.randn(B, T, H, 64, generator=g).to(cuda)
    gS = torch.randn(B, H, 64, 64, generator=g).to(cuda) * 0.1
    ref = _grads64(ins, gy, gS)
    S1 = ins[0].clone()
    hist = torch.empty(B, H, T, 64, 64, device=cuda)
    y1 = K.wkv7_f32(S1, *ins[1:], hist=hist)
    serial = [y1, S1, *K.wkv7_backward(hist, S1, *ins[1:], gy, gS)]
    chunked = [*K.dplr_seq_forward(*ins), *K.dplr_seq_backward(*ins, gy, gS)]
    for name, c, s, e in zip(("y", "S_T", "gS0", "gr", "gw", "gk", "gv", "ga", "gb"), chunked, serial, ref):
        assert _rel(c, e) <= 1.05 * _rel(s, e), f"{name}: {_rel(c, e):.3e} chunked, {_rel(s, e):.3e} serial"
    # 16-bit operands: the f32 state
    h = [x.half() for x in ins[1:]]
    S2, S3, S64 = ins[0].clone(), ins[0].clone(), ins[0].double()
    K.wkv7(S2, *h, chunked=True)
    K.wkv7(S3, *h, chunked=False)
    S64 = _grads64([S64, *h], gy, gS)[1]
    assert _rel(S2, S64) <= 1.05 * _rel(S3, S64), f"state: {_rel(S2, S64):.3e} chunked, {_rel(S3, S64):.3e} serial"


@pytest.mark.parametrize("which,scale", [(1, 1e-15), (3, 1e-15), (5, 1e-15), (1, 1e10), (3, 1e10)],
                         ids=["tiny_r", "tiny_k", "tiny_a", "large_r", "large_k"])
def test_chunked_f32_scans_keep_the_range_of_their_inputs(which, scale, cuda):
    """Decays whose products over a chunk come close to 1e-30 (0.016^16 = 2e-29)
    with inputs that leave f32's range when scaled by them: the chunked forward
    (146 tokens) and gradient (40) against 64 bits. fp32 sums of up to 64 + 146
    terms; measured below 2e-7, asserted at ten times that."""
    for T in (146, 40):
        ins = [x.to(cuda) for x in _dplr_inputs(1, T, 2, seed=T)]
        ins[2] = torch.full_like(ins[2], 0.016)
        ins[which] = ins[which] * scale
        gy = torch.randn(1, T, 2, 64, generator=torch.Generator().manual_seed(T)).to(cuda)
        ref = _grads64(ins, gy, torch.zeros_like(ins[0]))
        got = [*K.dplr_seq_forward(*ins), *K.dplr_seq_backward(*ins, gy, None)]
        for name, x, e in zip(("y", "S_T", "gS0", "gr", "gw", "gk", "gv", "ga", "gb"), got, ref):
            assert _rel(x, e) < 2e-6, f"T={T} {name}: {_rel(x, e):.2e}"


def _peak(fn):
    """fn() and the device bytes it took at most beyond what was held before."""
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    out = fn()
    torch.cuda.synchronize()
    return out, torch.cuda.max_memory_allocated() - base


@pytest.mark.parametrize("B,T,H,limit", [(5, 150, 3, 2), (2, 200, 2, 1), (1, 333, 2, 0.3), (3, 145, 1, 0.5)])
def test_chunked_scans_in_ranges_of_a_bounded_workspace(B, T, H, limit, cuda, monkeypatch):
    """A workspace of ``limit`` sequences' records: batches in parts, sequences in
    parts of whole chunks (the gradient: whole sequences), the same bits."""
    ins = [x.to(cuda) for x in _dplr_inputs(B, T, H, seed=T)]
    gy = torch.randn(B, T, H, 64, device=cuda)
    h = [x.half() for x in ins[1:]]

    def run():
        S = ins[0].clone()
        y = K.wkv7(S, *h, chunked=True)
        return [y, S, *K.dplr_seq_forward(*ins), *K.dplr_seq_backward(*ins, gy, None)]

    want = run()
    nb = int(K._lib.load().rwkv7_wkv7_chunked_workspace_bytes(1, T, H))
    monkeypatch.setattr(K, "CHUNK_WS_BYTES", int(limit * nb))
    for x, e in zip(run(), want):
        assert torch.equal(x, e)


def test_large_chunked_calls_keep_to_the_workspace_bound(cuda):
    """64 sequences x 2048 tokens x 32 heads, 7.6 GB of records in one piece:
    the call takes the bound and y beyond its operands."""
    B, T, H = 64, 2048, 32
    x = torch.randn(B, T, H, 64, device=cuda, dtype=torch.float16) * 0.1
    w = torch.full_like(x, 0.9)
    S = torch.zeros(B, H, 64, 64, device=cuda)
    y, peak = _peak(lambda: K.wkv7(S, x, w, x, x, x, x))
    assert peak <= K.CHUNK_WS_BYTES + y.numel() * 2 + (1 << 22)


@pytest.mark.parametrize("T", [1, 2, 3])
def test_gradient_of_a_few_tokens_of_many_heads(T, cuda):
    """384 heads of 1 to 3 tokens against 64 bits (fp32 sums of 64 terms and a few
    steps, 2e-6); one and two tokens take the recorded states, with no chunk
    workspace."""
    B, H = 24, 16
    ins = [x.to(cuda) for x in _dplr_inputs(B, T, H, seed=T)]
    g = torch.Generator().manual_seed(T)
    gy = torch.randn(B, T, H, 64, generator=g).to(cuda)
    gS = torch.randn(B, H, 64, 64, generator=g).to(cuda)
    ref = _grads64(ins, gy, gS)[2:]
    got, peak = _peak(lambda: K.dplr_seq_backward(*ins, gy, gS))
    for name, x, e in zip(("gS0", "gr", "gw", "gk", "gv", "ga", "gb"), got, ref):
        assert _rel(x, e) < 2e-6, f"{name}: {_rel(x, e):.2e}"
    records = int(K._lib.load().rwkv7_wkv7_grad_workspace_bytes(B, T, H))
    assert (peak < records) == (T <= 2)


@pytest.mark.parametrize("T", [119, 120, 127, 128, 143, 144])
@pytest.mark.parametrize("B", [1, 24], ids=["2_heads", "48_heads"])
def test_scans_around_the_lines_of_the_chunked_form(B, T, cuda):
    """Both sides of the lengths from which the operator and the training forward
    are chunked, against the serial scan (fp32 sums of 64 terms and 144 steps:
    below 1e-6 apart; f16 outputs to half a unit, 2^-11 of a value)."""
    ins = [x.to(cuda) for x in _dplr_inputs(B, T, 2, seed=T)]
    S1 = ins[0].clone()
    y1 = K.wkv7_f32(S1, *ins[1:])
    y, S_T = K.dplr_seq_forward(*ins)
    assert _rel(y, y1) < 1e-6 and _rel(S_T, S1) < 1e-6
    h = [x.half() for x in ins[1:]]
    S2, S3 = ins[0].clone(), ins[0].clone()
    y2, y3 = K.wkv7(S2, *h), K.wkv7(S3, *h, chunked=False)
    assert _rel(S2, S3) < 1e-6
    assert _rel(y2.float(), y3.float()) < 2**-11
