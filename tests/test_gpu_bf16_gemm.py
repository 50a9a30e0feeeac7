"""GPU parity of the bf16-weight projection path (bf16 configurations, e.g. C5 Llama-3-8B).

Two checks per op:
* tight: against the oracle's linear_f32_with_bias / SwiGLU / greedy head evaluated on the
  bf16-rounded operands (activations rounded to nearest even, weights widened exactly).  A
  product of two bf16 values is exact in f32, so only the summation order differs: 1e-5
  normwise.  This pins the packing, the MFMA fragment layout and the activation rounding;
* reference: against the reference semantics (f32 activations, weights widened from bf16 as
  io/safetensors.rs:540-542 loads them), within the bf16-storage tolerance 2e-2.
"""
import numpy as np
import pytest

from conftest import normwise_error

pytestmark = pytest.mark.gpu


def dev(x):
    import torch

    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def bf16_weights(rng, shape, scale=0.02):
    """Random weights as bf16 bits (RNE of N(0, scale))."""
    import oracle

    return oracle.f32_to_bf16((rng.standard_normal(shape, dtype=np.float32) * scale).astype(np.float32))


def round_bf16(orc, x):
    return orc.bf16_to_f32(orc.f32_to_bf16(x))


def sum_splits(parts):
    acc = parts[0].copy()
    for z in range(1, parts.shape[0]):
        acc = acc + parts[z]
    return acc


def padded(a):
    """Device copy of a [M, K] f32 array with rows padded to a multiple of 4 floats (NaN in the
    padding: the kernel must not read past K)."""
    import torch

    m, k = a.shape
    lda = (k + 3) // 4 * 4
    d = torch.full((m, lda), float("nan"), device="cuda")
    d[:, :k] = dev(a)
    return d[:, :k]


SHAPES = [  # (M, K, N): C5 decode / prefill tiles, C1 and C4 shapes, ragged tails; the C5 step's
    # M 2304 runs 128-row blocks over q|k|v's 24 column groups and 96-row blocks over 16 (K cut
    # short to keep the oracle quick)
    (256, 4096, 1024), (300, 512, 520), (64, 896, 1152), (8, 256, 688), (37, 96, 300),
    (1, 64, 40), (17, 100, 33), (130, 4096, 256), (5, 2, 3), (2304, 64, 6144), (2304, 96, 4096),
    (2300, 100, 4090),
]


@pytest.mark.parametrize("shape", SHAPES)
def test_bf16_gemm_matches_linear(orc, gpu_ctx, shape):
    import torch

    m, k, n = shape
    print(f"bf16 gemm shape={shape}", flush=True)
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    a = rng.standard_normal((m, k), dtype=np.float32)
    wb = bf16_weights(rng, (k, n))
    w = orc.bf16_to_f32(wb)
    bp = gpu_ctx.weight_pack_bf16(dev(wb.view(np.int16)), k, n)
    tight = orc.linear_with_bias(round_bf16(orc, a), w, None)
    ref = orc.linear_with_bias(a, w, None)
    for splits in sorted({1, 2, gpu_ctx.gemm_bf16_splits(m, k, n)}):
        q = (k + 31) // 32
        per = (q + splits - 1) // splits
        if (q + per - 1) // per != splits:
            continue
        out = torch.full((splits, m, n), float("nan"), device="cuda")
        gpu_ctx.gemm_bf16(padded(a), bp, k, n, splits, out)
        torch.cuda.synchronize()
        got = sum_splits(out.cpu().numpy())
        assert normwise_error(got, tight) <= 1e-5, (shape, splits)
        assert normwise_error(got, ref) <= 2e-2, (shape, splits)


def test_bf16_pack_sources_agree(gpu_ctx):
    """Packing from f32 (rounded on the device) equals packing the RNE bf16 bits; the column
    concatenation pack equals packing the concatenated matrix; the [N, K] source layout equals
    the transposed [K, N] one."""
    import torch

    import oracle

    rng = np.random.default_rng(7)
    k = 96
    parts = [(rng.standard_normal((k, n), dtype=np.float32) * 0.05).astype(np.float32) for n in (64, 16, 48)]
    cat = np.concatenate(parts, axis=1)
    bits = oracle.f32_to_bf16(cat).view(np.int16)
    p_f32 = gpu_ctx.weight_pack_bf16(dev(cat), k, 128)
    p_bits = gpu_ctx.weight_pack_bf16(dev(bits), k, 128)
    assert torch.equal(p_f32, p_bits)
    p_cols = gpu_ctx.weight_pack_bf16_columns([dev(p) for p in parts], k)
    assert torch.equal(p_cols, p_bits)
    p_t = gpu_ctx.weight_pack_bf16(dev(np.ascontiguousarray(bits.T)), k, 128, src_layout=1)
    assert torch.equal(p_t, p_bits)


@pytest.mark.parametrize("m,k,f,bias", [(8, 4096, 1024, False), (300, 256, 688, True), (64, 896, 4864, False),
                                        (3, 64, 40, True)])
def test_bf16_swiglu(orc, gpu_ctx, m, k, f, bias):
    import torch

    print(f"bf16 swiglu m={m} k={k} f={f}", flush=True)
    rng = np.random.default_rng(m + k + f)
    a = rng.standard_normal((m, k), dtype=np.float32)
    w1b, w3b = bf16_weights(rng, (k, f)), bf16_weights(rng, (k, f))
    w1, w3 = orc.bf16_to_f32(w1b), orc.bf16_to_f32(w3b)
    b1 = rng.standard_normal(f, dtype=np.float32) * 0.1 if bias else None
    b3 = rng.standard_normal(f, dtype=np.float32) * 0.1 if bias else None
    bp = gpu_ctx.weight_pack_bf16_pair(dev(w1b.view(np.int16)), dev(w3b.view(np.int16)), k, f)
    out = torch.full((m, f), float("nan"), device="cuda")
    gpu_ctx.gemm_bf16_swiglu(padded(a), bp, k, f, out, None if b1 is None else dev(b1),
                             None if b3 is None else dev(b3))
    torch.cuda.synchronize()
    got = out.cpu().numpy()

    def swiglu(x):
        up = orc.linear_with_bias(x, w1, b1)
        gate = orc.linear_with_bias(x, w3, b3)
        return orc.mul(up, orc.silu(gate))

    assert normwise_error(got, swiglu(round_bf16(orc, a))) <= 1e-5
    assert normwise_error(got, swiglu(a)) <= 2e-2


def logits_f64(hr, w, chunk=16384):
    """hr [M, H] times w [V, H]^T in f64, over vocabulary chunks (bounded host memory)."""
    out = np.empty((hr.shape[0], w.shape[0]), np.float64)
    h64 = hr.astype(np.float64)
    for v0 in range(0, w.shape[0], chunk):
        out[:, v0:v0 + chunk] = h64 @ w[v0:v0 + chunk].astype(np.float64).T
    return out


# (200, 256, 20000): 79 column groups over 96-row blocks (the third one partial), as the C5 head;
# (8, 4096, 128256): the C5 head itself (Llama-3-8B hidden and vocabulary)
@pytest.mark.parametrize("m,h,v", [(1, 64, 129), (4, 256, 4096), (257, 512, 3000), (8, 2048, 32000), (200, 256, 20000),
                                   (8, 4096, 128256)])
def test_bf16_lm_head_argmax(orc, gpu_ctx, m, h, v):
    import torch

    print(f"bf16 lm_head m={m} h={h} v={v}", flush=True)
    rng = np.random.default_rng(h + v)
    hid = rng.standard_normal((m, h), dtype=np.float32)
    wb = bf16_weights(rng, (v, h), 0.05)
    w = orc.bf16_to_f32(wb)
    bp = gpu_ctx.weight_pack_bf16(dev(wb.view(np.int16)), h, v, src_layout=1)
    del wb
    tok = torch.empty(m, dtype=torch.int32, device="cuda")
    prob = torch.empty(m, device="cuda")
    gpu_ctx.lm_head_argmax_bf16(padded(hid), bp, v, tok, prob)
    torch.cuda.synchronize()
    hr = round_bf16(orc, hid)
    logits = logits_f64(hr, w)
    rows = range(m) if m <= 64 else list(range(32)) + [m - 1]
    for r in rows:
        top2 = np.sort(logits[r])[-2:]
        if top2[1] - top2[0] < 1e-4 * max(1.0, abs(top2[1])):
            continue  # near tie: the summation order may pick the other index
        ridx, rprob = orc.matmul_rhs_transposed_argmax(hr[r:r + 1], w)
        assert int(tok[r]) == ridx, r
        assert abs(float(prob[r]) - rprob) <= 1e-4 * max(rprob, 1e-30) + 1e-7


def test_bf16_lm_head_reference_vector_and_ties(gpu_ctx):
    """matmul.rs:745-758: lhs [1,2], rhs [[1,0],[0,1],[1,1]] -> (2, 0.66524094) (all values
    exact in bf16); equal logits across slabs keep the first index."""
    import torch

    tok = torch.empty(1, dtype=torch.int32, device="cuda")
    prob = torch.empty(1, device="cuda")
    hid = torch.zeros((1, 4), device="cuda")
    hid[0, :2] = torch.tensor([1.0, 2.0])
    w = np.array([[1, 0], [0, 1], [1, 1]], np.float32)
    bp = gpu_ctx.weight_pack_bf16(dev(w), 2, 3, src_layout=1)
    gpu_ctx.lm_head_argmax_bf16(hid[:, :2], bp, 3, tok, prob)
    torch.cuda.synchronize()
    assert int(tok[0]) == 2
    assert abs(float(prob[0]) - 0.66524094) <= 1e-6
    v, h = 300, 4
    w = np.zeros((v, h), np.float32)
    w[[70, 5, 200, 71, 6], 0] = 1.0  # max logit 1.0 at 5, 6, 70, 71, 200 -> first is 5
    bp = gpu_ctx.weight_pack_bf16(dev(w), h, v, src_layout=1)
    gpu_ctx.lm_head_argmax_bf16(dev(np.array([[1, 0, 0, 0]], np.float32)), bp, v, tok, prob)
    torch.cuda.synchronize()
    assert int(tok[0]) == 5


def padded16(bits):
    """Device copy of [M, K] bf16 bits (uint16) with rows padded to a multiple of 8 elements (NaN
    bits in the padding: the kernel must not read past K)."""
    import torch

    m, k = bits.shape
    lda = (k + 7) // 8 * 8
    d = torch.full((m, lda), 0x7fc0, dtype=torch.int16, device="cuda")
    d[:, :k] = dev(bits.view(np.int16))
    return d[:, :k]


@pytest.mark.parametrize("shape", SHAPES)
def test_bf16_gemm_bf16_activations_bit_identical(orc, gpu_ctx, shape):
    """A handed over as bf16 bits (RNE of the f32 activations) gives exactly the f32 call's
    partials: the kernel rounds f32 activations with the same rule."""
    import torch

    m, k, n = shape
    print(f"bf16-activation gemm shape={shape}", flush=True)
    rng = np.random.default_rng(5 * m + k + n)
    a = rng.standard_normal((m, k), dtype=np.float32)
    wb = bf16_weights(rng, (k, n))
    bp = gpu_ctx.weight_pack_bf16(dev(wb.view(np.int16)), k, n)
    splits = gpu_ctx.gemm_bf16_splits(m, k, n)
    ref = torch.full((splits, m, n), float("nan"), device="cuda")
    got = torch.full((splits, m, n), float("nan"), device="cuda")
    gpu_ctx.gemm_bf16(padded(a), bp, k, n, splits, ref)
    gpu_ctx.gemm_bf16(padded16(orc.f32_to_bf16(a)), bp, k, n, splits, got)
    torch.cuda.synchronize()
    assert torch.equal(got, ref), shape


@pytest.mark.parametrize("m,k,f", [(300, 256, 688), (2304, 4096, 1024), (64, 896, 4864), (3, 100, 40)])
def test_bf16_swiglu_bf16_in_out(orc, gpu_ctx, m, k, f):
    """bf16 activations in: the same f32 output as the f32 call; bf16 output: exactly the RNE
    of the f32 output (direct epilogue and the split-sum path alike)."""
    import torch

    print(f"bf16 swiglu bf16 in/out m={m} k={k} f={f}", flush=True)
    rng = np.random.default_rng(m * 7 + k + f)
    a = rng.standard_normal((m, k), dtype=np.float32)
    w1b, w3b = bf16_weights(rng, (k, f)), bf16_weights(rng, (k, f))
    bp = gpu_ctx.weight_pack_bf16_pair(dev(w1b.view(np.int16)), dev(w3b.view(np.int16)), k, f)
    b1 = dev(rng.standard_normal(f, dtype=np.float32) * 0.1)
    out32 = torch.full((m, f), float("nan"), device="cuda")
    gpu_ctx.gemm_bf16_swiglu(padded(a), bp, k, f, out32, b1, None)
    a16 = padded16(orc.f32_to_bf16(a))
    out32b = torch.full((m, f), float("nan"), device="cuda")
    gpu_ctx.gemm_bf16_swiglu(a16, bp, k, f, out32b, b1, None)
    out16 = torch.full((m, f), 0x7fc0, dtype=torch.int16, device="cuda")
    gpu_ctx.gemm_bf16_swiglu(a16, bp, k, f, out16, b1, None)
    torch.cuda.synchronize()
    assert torch.equal(out32b, out32)
    want = orc.f32_to_bf16(out32.cpu().numpy())
    assert np.array_equal(out16.cpu().numpy().view(np.uint16), want)


@pytest.mark.parametrize("m,h,v", [(33, 200, 1000), (8, 4096, 128256)])
def test_bf16_head_bf16_activations(orc, gpu_ctx, m, h, v):
    """The greedy head over bf16 activations: the f32 call's tokens and probabilities exactly
    (also at the C5 head, 4096 -> 128256); at the C5 head the tokens also match the oracle's
    fused argmax over the bf16-rounded rows (matmul.rs:190-274) away from near ties."""
    import torch

    print(f"bf16 head bf16 activations m={m} h={h} v={v}", flush=True)
    rng = np.random.default_rng(21 + v)
    hid = rng.standard_normal((m, h), dtype=np.float32)
    wb = bf16_weights(rng, (v, h))
    bp = gpu_ctx.weight_pack_bf16(dev(wb.view(np.int16)), h, v, src_layout=1)
    tok = [torch.empty(m, dtype=torch.int32, device="cuda") for _ in range(2)]
    prob = [torch.empty(m, device="cuda") for _ in range(2)]
    gpu_ctx.lm_head_argmax_bf16(padded(hid), bp, v, tok[0], prob[0])
    gpu_ctx.lm_head_argmax_bf16(padded16(orc.f32_to_bf16(hid)), bp, v, tok[1], prob[1])
    torch.cuda.synchronize()
    assert torch.equal(tok[0], tok[1]) and torch.equal(prob[0], prob[1])
    if v < 100000:
        return
    w = orc.bf16_to_f32(wb)
    del wb
    hr = round_bf16(orc, hid)
    logits = logits_f64(hr, w)
    for r in range(m):
        top2 = np.sort(logits[r])[-2:]
        if top2[1] - top2[0] < 1e-4 * max(1.0, abs(top2[1])):
            continue
        ridx, rprob = orc.matmul_rhs_transposed_argmax(hr[r:r + 1], w)
        assert int(tok[1][r]) == ridx, r
        assert abs(float(prob[1][r]) - rprob) <= 1e-4 * max(rprob, 1e-30) + 1e-7


@pytest.mark.parametrize("n,offset", [(1, 0), (7, 0), (4096 * 37 + 3, 0), (1000, 1), (1 << 20, 0)])
def test_convert_f32_to_bf16(orc, gpu_ctx, n, offset):
    """fi_convert_f32_to_bf16 against the oracle's nearest-even narrowing, with ties, the
    largest finite values, infinities, NaN, denormals and signed zeros; an offset start
    exercises the unaligned path."""
    import torch

    rng = np.random.default_rng(n)
    x = rng.standard_normal(n + offset, dtype=np.float32) * np.float32(100)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 3.4028235e38, -3.4028235e38, 1e-40, -1e-41,
                        1.00390625, 1.01171875, -1.00390625], np.float32)  # ties: 1 + 2^-8, 1 + 3 * 2^-8
    x[offset:offset + min(n, special.size)] = special[:min(n, special.size)]
    src = dev(x)[offset:]
    out = torch.full((n + 1,), 0x1234, dtype=torch.int16, device="cuda")
    gpu_ctx.convert_f32_to_bf16(src, out[:n])
    torch.cuda.synchronize()
    got = out.cpu().numpy().view(np.uint16)
    want = orc.f32_to_bf16(x[offset:])
    nan = np.isnan(x[offset:])
    assert np.array_equal(got[:n][~nan], want[~nan])
    assert np.all((got[:n][nan] & 0x7f80) == 0x7f80) and np.all((got[:n][nan] & 0x7f) != 0)
    assert got[n] == 0x1234  # nothing written past n


@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("k,n", [(24, 4090), (1000, 4112), (4864, 896), (520, 8200), (1001, 4112), (525, 896),
                                 (31, 8200)])
def test_bf16_few_rows_edges(gpu_ctx, m, k, n):
    """Both sides of every row-tile and slab-count choice up to 64 rows (and the first row count
    past it), K shorter than one step, with a tail, an uneven last part and several stages:
    partials and SwiGLU against f64 on the same bf16 operands.  Products are exact in f32, so
    only the f32 sums differ: 1e-5 normwise; f32 and bf16 activations agree bit for bit."""
    import torch

    print(f"bf16 few rows m={m} k={k} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    normal = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    a16 = torch.full((m, (k + 7) // 8 * 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    a16[:, :k] = normal(m, k)
    a32 = a16.float()
    w, w3 = (normal(k, n) * 0.02).bfloat16(), (normal(k, n) * 0.02).bfloat16()
    exact = a16[:, :k].double() @ w.double()
    bp, pair = gpu_ctx.weight_pack_bf16(w, k, n), gpu_ctx.weight_pack_bf16_pair(w, w3, k, n)

    def err(got, want):
        return ((got.double() - want).norm() / want.norm()).item()

    for splits in sorted({1, gpu_ctx.gemm_bf16_splits(m, k, n)}):
        parts = [torch.full((splits, m, n), float("nan"), device="cuda") for _ in range(2)]
        for a, out in zip((a16, a32), parts):
            gpu_ctx.gemm_bf16(a[:, :k], bp, k, n, splits, out)
        assert torch.equal(parts[0], parts[1])
        assert err(parts[0].sum(dim=0), exact) <= 1e-5, splits
    act = [torch.full((m, n), float("nan"), device="cuda") for _ in range(2)]
    for a, out in zip((a16, a32), act):
        gpu_ctx.gemm_bf16_swiglu(a[:, :k], pair, k, n, out)
    assert torch.equal(act[0], act[1])
    assert err(act[0], exact * torch.nn.functional.silu(a16[:, :k].double() @ w3.double())) <= 1e-5


@pytest.mark.parametrize("rows", [1, 256, 257])
def test_residual_norm_wide_rows(gpu_ctx, rows):
    """Rows of 2048 columns and more, on both sides of the row count that takes wide workgroups,
    against f64; 4101 columns take the scalar loop."""
    import torch

    for hidden in (2048, 4096, 4101, 33000):
        print(f"wide residual norm rows={rows} hidden={hidden}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(rows + hidden)
        normal = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
        parts, res, w = normal(3, rows, hidden), normal(rows, hidden), normal(hidden)
        total, out = torch.empty_like(res), torch.empty_like(res)
        gpu_ctx.splitk_residual_rms_norm(parts, 3, None, res, total, w, out, 1e-6)
        want = parts.double().sum(dim=0) + res.double()
        normed = want / (want.square().mean(dim=1, keepdim=True) + 1e-6).sqrt() * w.double()
        for got, exact in ((total, want), (out, normed)):
            assert ((got.double() - exact).norm() / exact.norm()).item() <= 1e-6


@pytest.mark.parametrize("hidden", [2048, 4096, 4100, 4101, 8192, 12292, 32768, 32772])
def test_residual_norm_row_bits_do_not_depend_on_row_count(gpu_ctx, hidden):
    """Calls of up to one row a CU take wide workgroups, larger ones narrow workgroups: a row of
    the same partials has the same bits in both, f32 and bf16, with and without a bias."""
    import torch

    print(f"residual norm row bits hidden={hidden}", flush=True)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator(device="cuda").manual_seed(hidden)
    normal = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    n = cus + 1
    parts, res, w, bias = normal(2, n, hidden), normal(n, hidden), normal(hidden), normal(hidden)

    def run(rows, dtype, b):
        total, out = torch.empty(rows, hidden, device="cuda"), torch.empty(rows, hidden, device="cuda", dtype=dtype)
        gpu_ctx.splitk_residual_rms_norm(parts[:, :rows].contiguous(), 2, b, res[:rows].contiguous(), total, w, out,
                                         1e-6)
        return total, out

    for dtype in (torch.float32, torch.bfloat16):
        for b in (None, bias):
            whole = run(n, dtype, b)
            for rows in (1, 33, cus):
                for few, many in zip(run(rows, dtype, b), whole):
                    assert torch.equal(few, many[:rows]), (dtype, rows)


@pytest.mark.parametrize("m,k,n", [
    (1, 4096, 256), (16, 2050, 1024), (48, 1024, 256),     # few slabs behind a long K: split
    (64, 1024, 4592), (64, 1024, 4608), (33, 4101, 4800),  # both sides of the slabs that fill the chip
    (16, 64, 8192), (17, 520, 8208),                       # both sides of four slabs a CU
    (64, 5728, 8208), (64, 5760, 8208)])                   # more slabs, both sides of the longest chain
def test_bf16_swiglu_few_rows_route(gpu_ctx, m, k, n):
    """SwiGLU of up to 64 rows on both sides of each choice (one launch over all of K, of four or
    eight slabs a workgroup, or row tiles with K split): against f64 on the same bf16 operands,
    whose products are exact in f32, so only the f32 sums differ (1e-5 normwise); f32 and bf16 rows
    agree bit for bit; with biases, and into bf16, which is the f32 result rounded to nearest even."""
    import torch

    print(f"bf16 swiglu route m={m} k={k} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    normal = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    a16 = torch.full((m, (k + 7) // 8 * 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    a16[:, :k] = normal(m, k)
    w1, w3 = (normal(k, n) * 0.02).bfloat16(), (normal(k, n) * 0.02).bfloat16()
    bias = normal(2, n) * 0.1
    pair = gpu_ctx.weight_pack_bf16_pair(w1, w3, k, n)
    x = a16[:, :k].double()
    up, gate = x @ w1.double(), x @ w3.double()
    for b in ((None, None), (bias[0], bias[1])):
        outs = []
        for a in (a16, a16.float()):
            outs.append(torch.full((m, n), float("nan"), device="cuda"))
            gpu_ctx.gemm_bf16_swiglu(a[:, :k], pair, k, n, outs[-1], *b)
        assert torch.equal(outs[0], outs[1])
        want = up * torch.nn.functional.silu(gate) if b[0] is None else \
            (up + bias[0].double()) * torch.nn.functional.silu(gate + bias[1].double())
        assert ((outs[0].double() - want).norm() / want.norm()).item() <= 1e-5
        narrow = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
        gpu_ctx.gemm_bf16_swiglu(a16[:, :k], pair, k, n, narrow, *b)
        assert torch.equal(narrow, outs[0].bfloat16())


@pytest.mark.parametrize("n", [32768, 32784, 65536, 65552])
@pytest.mark.parametrize("m,k", [(1, 72), (16, 2047), (16, 2048), (17, 2048), (17, 2049), (32, 40), (33, 72), (64, 40)])
def test_bf16_wide_few_rows_route(gpu_ctx, m, k, n):
    """Wide products of up to 64 rows (a head's logits) on both sides of each choice between the
    two kernels, in one split and in the library's count, against f64 on the same bf16 operands
    (1e-5 normwise: only f32 sums differ); f32 and bf16 rows agree bit for bit."""
    import torch

    print(f"bf16 wide few rows m={m} k={k} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    a16 = torch.full((m, (k + 7) // 8 * 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    a16[:, :k] = torch.randn(m, k, generator=g, device="cuda")
    w = (torch.randn(k, n, generator=g, device="cuda") * 0.02).bfloat16()
    want = a16[:, :k].double() @ w.double()
    bp = gpu_ctx.weight_pack_bf16(w, k, n)
    for splits in sorted({1, gpu_ctx.gemm_bf16_splits(m, k, n)}):
        outs = []
        for a in (a16, a16.float()):
            outs.append(torch.full((splits, m, n), float("nan"), device="cuda"))
            gpu_ctx.gemm_bf16(a[:, :k], bp, k, n, splits, outs[-1])
        assert torch.equal(outs[0], outs[1])
        assert ((outs[0].double().sum(dim=0) - want).norm() / want.norm()).item() <= 1e-5


@pytest.mark.parametrize("k,n", [(256, 688), (896, 4864), (4096, 4096), (4096, 14336), (14336, 4096)])
def test_bf16_few_rows_are_as_exact_as_many(gpu_ctx, k, n):
    """Products are exact in f32, so a kernel's distance from 64 bits is that of its f32 sums: with
    up to 64 rows no further off than the same rows in a call of 65, which takes row tiles.  5 %
    more is left for the spread of the mean over at least 16 x 688 values (about 1 %)."""
    import torch

    print(f"bf16 few rows exactness k={k} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(k + n)
    a = torch.randn(65, k, generator=g, device="cuda").bfloat16()
    w1, w3 = ((torch.randn(k, n, generator=g, device="cuda") * 0.02).bfloat16() for _ in range(2))
    up, gate = a.double() @ w1.double(), a.double() @ w3.double()
    want = up, up * torch.nn.functional.silu(gate)
    bp, pair = gpu_ctx.weight_pack_bf16(w1, k, n), gpu_ctx.weight_pack_bf16_pair(w1, w3, k, n)

    def run(m):
        splits = gpu_ctx.gemm_bf16_splits(m, k, n)
        parts, act = torch.empty(splits, m, n, device="cuda"), torch.empty(m, n, device="cuda")
        gpu_ctx.gemm_bf16(a[:m], bp, k, n, splits, parts)
        gpu_ctx.gemm_bf16_swiglu(a[:m], pair, k, n, act)
        total = parts[0].clone()
        for p in parts[1:]:  # f32, in split order, as the consumers add them
            total += p
        return total, act

    many = run(65)
    for m in (16, 32, 64):
        for few, ref, exact in zip(run(m), many, want):
            off = [(x[:m].double() - exact[:m]).norm().item() for x in (few, ref)]
            assert off[0] <= 1.05 * off[1], (m, off)
