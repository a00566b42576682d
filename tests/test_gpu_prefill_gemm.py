"""K6 (csrc/prefill_gemm.hip): the prompt projections with the RMSNorm prologue and the SwiGLU /
residual epilogues, against fp64 references of the same split-activation products, across
row / column tails, both activation layouts and every preset's shapes."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def K():
    from mdlarc_scale_amd import kernels

    return kernels


def split(v: torch.Tensor):
    hi = v.to(torch.bfloat16)
    return hi, (v - hi.float()).to(torch.bfloat16)


def rel(a: torch.Tensor, b: torch.Tensor) -> float:
    return ((a.double() - b.double()).abs().max() / b.double().abs().max()).item()


# (m, n, k): row tails (m % 256), column tails (n % 256), every preset's K (d, d_ff)
SHAPES = [(1000, 768, 768), (333, 1408, 256), (4097, 2304, 768), (17, 768, 2048),
          (700, 1280, 3392), (256, 3072, 1024), (1, 256, 704), (1025, 4096, 2752)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_split_gemm_matches_fp64(m, n, k):
    """out = (hi + lo) . W^T to fp32 accumulation error, identical in both activation layouts."""
    g = torch.Generator().manual_seed(m + n + k)
    w = (0.05 * torch.randn(n, k, generator=g)).to(torch.bfloat16).to(DEV)
    hi, lo = split(torch.randn(m, k, generator=g).to(DEV))
    a = torch.cat([hi, lo], 1).contiguous()
    ref = (hi.double() + lo.double()) @ w.double().t()
    wt = K().tile_matrix(w)
    out = torch.full((m, n), float("nan"), device=DEV)
    K().prefill_gemm_split(a, wt, out, k)
    out_t = torch.full((m, n), float("nan"), device=DEV)
    K().prefill_gemm_split(K().tile_matrix(a), wt, out_t, k, a_tiled=True)
    torch.cuda.synchronize()
    assert rel(out, ref) < 2e-6
    assert torch.equal(out, out_t)


@pytest.mark.parametrize("m,n,k", [s for s in SHAPES if s[2] <= 2048])
def test_norm_gemm_matches_fp64(m, n, k):
    """The ln1 + qkv form: split(x * gamma) . W^T (x * gamma rounded to fp32, then split) and
    rstd = 1 / sqrt(mean(x^2) + eps)."""
    g = torch.Generator().manual_seed(7 * m + n + k)
    w = (0.05 * torch.randn(n, k, generator=g)).to(torch.bfloat16).to(DEV)
    x = torch.randn(m, k, generator=g).to(DEV)
    gam = (1 + 0.1 * torch.randn(k, generator=g)).to(DEV)
    th, tl = split(x * gam)
    ref = (th.double() + tl.double()) @ w.double().t()
    rs_ref = 1 / torch.sqrt((x.double() ** 2).mean(1) + 1e-5)
    out = torch.empty(m, n, device=DEV)
    rs = torch.empty(m, device=DEV)
    K().prefill_gemm_norm(K().tile_f32(x), gam, 1e-5, K().tile_matrix(w), out, rs, k)
    torch.cuda.synchronize()
    assert rel(out, ref) < 2e-6
    assert rel(rs, rs_ref) < 1e-6


@pytest.mark.parametrize("m,n,k", [s for s in SHAPES if s[1] % 32 == 0])
@pytest.mark.parametrize("bias", [False, True])
def test_residual_gemm_matches_fp64(m, n, k, bias):
    """x += (hi + lo) . W^T (+ bias) in place on the fp32 tile-layout residual stream; both
    activation layouts give the same x; padding rows of the tile buffer are left alone."""
    g = torch.Generator().manual_seed(3 * m + n + k + bias)
    w = (0.05 * torch.randn(n, k, generator=g)).to(torch.bfloat16).to(DEV)
    hi, lo = split(torch.randn(m, k, generator=g).to(DEV))
    a = torch.cat([hi, lo], 1).contiguous()
    x0 = torch.randn(m, n, generator=g).to(DEV)
    b = torch.randn(n, generator=g).to(DEV) if bias else None
    ref = x0.double() + (hi.double() + lo.double()) @ w.double().t()
    if bias:
        ref += b.double()
    wt = K().tile_matrix(w)
    x1 = K().tile_f32(x0)
    x1_before = x1.clone()
    K().prefill_gemm_split_residual(a, wt, x1, b, m, n, k)
    x2 = K().tile_f32(x0)
    K().prefill_gemm_split_residual(K().tile_matrix(a), wt, x2, b, m, n, k, a_tiled=True)
    torch.cuda.synchronize()
    assert rel(K().untile_f32(x1, m, n), ref) < 2e-6
    assert torch.equal(x1, x2)
    # the tile buffer's padding rows (m .. tile_rows(m) - 1) keep their values
    untiled = lambda t: K().untile_f32(t, K().tile_rows(m), n)  # noqa: E731
    assert torch.equal(untiled(x1)[m:], untiled(x1_before)[m:])


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("m,f,k", [(1000, 2048, 768), (333, 704, 256), (257, 2752, 1024),
                                   (700, 3392, 1280), (5, 2048, 768)])
def test_norm_swiglu_gemm(m, f, k, bias):
    """The ln2 + gate/up + SwiGLU form equals K3 (mdl_swiglu) applied to the same launch's gate /
    up accumulators (the E_STORE form on the interleaved weight, same main loop), bit for bit;
    and an fp64 reference to fp32 rounding.  Without biases (NULL) the epilogue adds zeros."""
    g = torch.Generator().manual_seed(m + f + k)
    wg = (0.05 * torch.randn(f, k, generator=g)).to(torch.bfloat16).to(DEV)
    wu = (0.05 * torch.randn(f, k, generator=g)).to(torch.bfloat16).to(DEV)
    wgu = K().tile_matrix(K().interleave_gate_up(wg, wu))
    x = torch.randn(m, k, generator=g).to(DEV)
    gam = (1 + 0.1 * torch.randn(k, generator=g)).to(DEV)
    bg = torch.randn(f, generator=g).to(DEV)
    bu = torch.randn(f, generator=g).to(DEV)
    if not bias:
        bg = bu = None
    xt = K().tile_f32(x)
    h = torch.empty(K().split_numel(m, f, True), dtype=torch.bfloat16, device=DEV)
    K().prefill_gemm_norm_swiglu(xt, gam, 1e-5, wgu, bg, bu, h, m, f, k)
    # unfused: gate / up accumulators (interleaved 16-column blocks) + rstd, then K3
    acc = torch.empty(m, 2 * f, device=DEV)
    rs = torch.empty(m, device=DEV)
    K().prefill_gemm_norm(xt, gam, 1e-5, wgu, acc, rs, k)
    blocks = acc.view(m, f // 16, 2, 16)
    gu = torch.cat([blocks[:, :, 0].reshape(m, f), blocks[:, :, 1].reshape(m, f)], 1).contiguous()
    h_ref = torch.empty(m, 2 * f, dtype=torch.bfloat16, device=DEV)
    K().swiglu(gu, rs, bg, bu, h_ref)
    torch.cuda.synchronize()
    assert torch.equal(K().untile_matrix(h, m, 2 * f), h_ref)
    th, tl = split(x * gam)
    t = th.double() + tl.double()
    rs64 = 1 / torch.sqrt((x.double() ** 2).mean(1) + 1e-5)
    gg = rs64[:, None] * (t @ wg.double().t())
    uu = rs64[:, None] * (t @ wu.double().t())
    if bias:
        gg, uu = gg + bg.double(), uu + bu.double()
    ref = gg / (1 + torch.exp(-gg)) * uu
    hh = K().untile_matrix(h, m, 2 * f).double()
    assert rel(hh[:, :f] + hh[:, f:], ref) < 2e-5


@pytest.mark.parametrize("m,n,k", [s for s in SHAPES if s[1] % 32 == 0])
def test_hi_only_split_forms_match_fp64(m, n, k):
    """a_parts 1: a holds hi alone ([m, k]) and the product is hi . W^T -- against fp64 to fp32
    accumulation error, in both layouts and both epilogues, and measurably apart from the split
    product (so a kernel that still added a lo term, or dropped hi, fails)."""
    g = torch.Generator().manual_seed(5 * m + n + k)
    w = (0.05 * torch.randn(n, k, generator=g)).to(torch.bfloat16).to(DEV)
    v = torch.randn(m, k, generator=g).to(DEV)
    hi, lo = split(v)
    a = hi.contiguous()
    ref = hi.double() @ w.double().t()
    assert rel(v.double() @ w.double().t(), ref) > 1e-4   # the lo term matters at this scale
    wt = K().tile_matrix(w)
    out = torch.full((m, n), float("nan"), device=DEV)
    K().prefill_gemm_split(a, wt, out, k, a_parts=1)
    out_t = torch.full((m, n), float("nan"), device=DEV)
    K().prefill_gemm_split(K().tile_matrix(a), wt, out_t, k, a_tiled=True, a_parts=1)
    x0 = torch.randn(m, n, generator=g).to(DEV)
    b = torch.randn(n, generator=g).to(DEV)
    x1 = K().tile_f32(x0)
    K().prefill_gemm_split_residual(K().tile_matrix(a), wt, x1, b, m, n, k, a_tiled=True,
                                    a_parts=1)
    x2 = K().tile_f32(x0)
    K().prefill_gemm_split_residual(a, wt, x2, b, m, n, k, a_parts=1)
    torch.cuda.synchronize()
    assert rel(out, ref) < 2e-6
    assert torch.equal(out, out_t)
    assert rel(K().untile_f32(x1, m, n), x0.double() + ref + b.double()) < 2e-6
    assert torch.equal(x1, x2)


@pytest.mark.parametrize("m,f,k", [(1000, 2048, 768), (333, 704, 256), (257, 2752, 1024),
                                   (5, 2048, 768)])
def test_norm_swiglu_parts(m, f, k):
    """a_parts 1 (gate / up of bf16(x * gamma)) against fp64 of the same hi product, h_parts 1
    (hi of h alone, [m, f]) bit-equal to the hi half of the h_parts 2 output of the same launch
    form, for both activation forms."""
    g = torch.Generator().manual_seed(3 * m + f + k)
    wg = (0.05 * torch.randn(f, k, generator=g)).to(torch.bfloat16).to(DEV)
    wu = (0.05 * torch.randn(f, k, generator=g)).to(torch.bfloat16).to(DEV)
    wgu = K().tile_matrix(K().interleave_gate_up(wg, wu))
    x = torch.randn(m, k, generator=g).to(DEV)
    gam = (1 + 0.1 * torch.randn(k, generator=g)).to(DEV)
    bg = torch.randn(f, generator=g).to(DEV)
    bu = torch.randn(f, generator=g).to(DEV)
    xt = K().tile_f32(x)
    hs = {}
    for ap in (1, 2):
        for hp in (1, 2):
            h = torch.empty(K().tile_rows(m) * hp * f, dtype=torch.bfloat16, device=DEV)
            K().prefill_gemm_norm_swiglu(xt, gam, 1e-5, wgu, bg, bu, h, m, f, k, a_parts=ap,
                                         h_parts=hp)
            hs[ap, hp] = K().untile_matrix(h, m, hp * f)
    torch.cuda.synchronize()
    for ap in (1, 2):
        assert torch.equal(hs[ap, 1], hs[ap, 2][:, :f])
    th, tl = split(x * gam)
    rs64 = 1 / torch.sqrt((x.double() ** 2).mean(1) + 1e-5)

    def swiglu64(t):
        gg = rs64[:, None] * (t @ wg.double().t()) + bg.double()
        uu = rs64[:, None] * (t @ wu.double().t()) + bu.double()
        return gg / (1 + torch.exp(-gg)) * uu

    ref_hi, ref_split = swiglu64(th.double()), swiglu64(th.double() + tl.double())
    h12 = hs[1, 2].double()
    assert rel(h12[:, :f] + h12[:, f:], ref_hi) < 2e-5
    assert rel(ref_split, ref_hi) > 1e-4   # the lo term is visible at this tolerance


def test_prefill_gemm_persistent_tiles_cover_everything():
    """More tiles than CUs (each block walks several, the load ring crossing tile boundaries):
    every output element is written once with the right value."""
    g = torch.Generator().manual_seed(11)
    m, n, k = 256 * 70 + 19, 2304, 256      # 639 tiles: each of the <= 256 blocks walks 2-3
    w = (0.05 * torch.randn(n, k, generator=g)).to(torch.bfloat16).to(DEV)
    hi, lo = split(torch.randn(m, k, generator=g).to(DEV))
    a = torch.cat([hi, lo], 1).contiguous()
    out = torch.full((m, n), float("nan"), device=DEV)
    K().prefill_gemm_split(a, K().tile_matrix(w), out, k)
    ref = (hi.double() + lo.double()) @ w.double().t()
    torch.cuda.synchronize()
    assert not bool(out.isnan().any())
    assert rel(out, ref) < 2e-6


def _rope(max_xyz=(30, 30, 8)):
    from mdlarc_scale_amd.transformer import RotaryEmbedding3D

    rope = RotaryEmbedding3D(64, *max_xyz)
    return rope.device_table(DEV), (rope.max_x, rope.max_y, rope.max_z, rope.px, rope.py, rope.pz)


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("n_heads", [4, 12])
def test_norm_qkv_equals_norm_gemm_then_k2(packed, n_heads):
    """ln1 + qkv_proj + K2 in one launch writes exactly what the E_STORE form followed by K2
    (qkv_rope_cache / _packed) writes -- q, every cache slot, rstd -- and the fp32 projection
    rows only for each row's first LEAD_QUERIES tokens from kv_start."""
    g = torch.Generator().manual_seed(n_heads * 2 + packed)
    B, S, slots = 3, 150, 170
    H, d = n_heads, 64 * n_heads
    kv = [0, 37, 149]
    if packed:   # valid tokens of each row, then one padding token (slot -1, no cache write)
        tr, ts = [], []
        for b, k0 in enumerate(kv):
            tr += [b] * (S - k0)
            ts += list(range(k0, S))
        tr.append(1)
        ts.append(-1)
        rows = len(tr)
        token_row = torch.tensor(tr, dtype=torch.int32, device=DEV)
        token_slot = torch.tensor(ts, dtype=torch.int32, device=DEV)
    else:
        rows = B * S
        token_row = token_slot = None
    x = torch.randn(rows, d, generator=g).to(DEV)
    gam = (1 + 0.1 * torch.randn(d, generator=g)).to(DEV)
    w = K().tile_matrix((0.05 * torch.randn(3 * d, d, generator=g)).to(torch.bfloat16).to(DEV))
    pos = torch.randint(0, 35, (rows, 3), generator=g).to(DEV)
    tab, geom = _rope()
    kv_dev = torch.tensor(kv, dtype=torch.int32, device=DEV)
    xt = K().tile_f32(x)
    # reference: E_STORE form, then K2
    qkv = torch.empty(rows, 3 * d, device=DEV)
    rs1 = torch.empty(rows, device=DEV)
    K().prefill_gemm_norm(xt, gam, 1e-5, w, qkv, rs1, d)
    sentinel = torch.full((B, H, slots, 64), 7.0, dtype=torch.bfloat16)
    kc1, vc1 = sentinel.clone().to(DEV), sentinel.clone().to(DEV)
    q1 = torch.empty(rows, d, dtype=torch.bfloat16, device=DEV)
    if packed:
        K().qkv_rope_cache_packed(qkv, rs1, pos, tab, geom, token_row, token_slot, H, 0.125, q1,
                                  kc1, vc1)
    else:
        K().qkv_rope_cache(qkv, rs1, pos, tab, geom, B, S, H, 0.125, q1, kc1, vc1, slot0=0)
    # fused
    kc2, vc2 = sentinel.clone().to(DEV), sentinel.clone().to(DEV)
    q2 = torch.empty(rows, d, dtype=torch.bfloat16, device=DEV)
    rs2 = torch.empty(rows, device=DEV)
    lead = torch.full((rows, 3 * d), float("nan"), device=DEV)
    K().prefill_gemm_norm_qkv(xt, gam, 1e-5, w, rows, H, rs2, lead, K().LEAD_QUERIES, kv_dev, pos,
                              tab, geom, 0.125, q2, kc2, vc2, token_row=token_row,
                              token_slot=token_slot, seq=0 if packed else S)
    torch.cuda.synchronize()
    assert torch.equal(rs1, rs2)
    assert torch.equal(q1, q2)
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    # lead rows: slot in [kv_start[b], kv_start[b] + 64)
    if packed:
        rb, sl = token_row.long().cpu(), token_slot.long().cpu()
    else:
        rb = torch.arange(rows) // S
        sl = torch.arange(rows) % S
    ks = torch.tensor(kv)[rb]
    is_lead = (sl >= ks) & (sl - ks < K().LEAD_QUERIES)
    assert int(is_lead.sum()) > 0
    li = is_lead.to(DEV)
    assert torch.equal(lead[li], qkv[li])
    assert bool(lead[~li].isnan().all())


def test_split_gemm_at_config2_size_against_hipblaslt():
    """At config 2's packed prefill size (268,148 rows, the qkv projection's N = 2304, K = 768)
    K6 agrees with hipBLASLt on the [W | W] operand (an independent GEMM, fp32 accumulation in
    another order) to fp32 rounding over every element, and with fp64 on sampled rows."""
    from mdlarc_scale_amd.engine import gemm_f32, pack_split_weight

    g = torch.Generator(device=DEV).manual_seed(3)
    m, n, k = 268_148, 2304, 768
    w = (0.05 * torch.randn(n, k, generator=g, device=DEV)).to(torch.bfloat16)
    v = torch.randn(m, k, generator=g, device=DEV)
    hi, lo = split(v)
    a = torch.cat([hi, lo], 1).contiguous()
    del v, lo
    out = torch.empty(m, n, device=DEV)
    K().prefill_gemm_split(K().tile_matrix(a), K().tile_matrix(w), out, k, a_tiled=True)
    ref = torch.empty(m, n, device=DEV)
    gemm_f32(a, pack_split_weight(w, DEV), ref)
    torch.cuda.synchronize()
    scale = ref.abs().max()
    assert float((out - ref).abs().max() / scale) < 2e-6
    rows = torch.randint(0, m, (512,), generator=g, device=DEV)
    aa = a[rows].double()
    sub = (aa[:, :k] + aa[:, k:]) @ w.double().t()
    assert float((out[rows].double() - sub).abs().max() / sub.abs().max()) < 2e-6


# rows at the tiles' edges, and where products of d = 768 change their block shape
ROUTE_ROWS = [1, 63, 65, 257, 731, 1025, 2047, 3000, 4097, 6030, 8193]
MANY_ROWS = 20_600       # the shape of the largest gate / up products, from 20,481 rows on
MANY_QKV_ROWS = 36_400   # the same of qkv, from 36,353
F32W_ROWS = [1, 17, 250, 641, 768, 769, 1025, 1500, 2048, 2049, 3000, 4097, 8193]   # K5 up to 768
F32W_QKV_ROWS = [1, 448, 449, 640, 641, 1100, 4097, 12345]              # K5 up to 448


@pytest.mark.parametrize("form,n,k,rows", [
    ("NORM", 4096, 768, ROUTE_ROWS + [MANY_ROWS]), ("SPLIT", 768, 768, ROUTE_ROWS + [MANY_ROWS]),
    ("NORM", 2304, 768, ROUTE_ROWS + [MANY_QKV_ROWS]),
    ("NORM_F32W", 1408, 768, [m for m in F32W_ROWS if m > 768]),
    ("SPLIT_F32W", 768, 768, [m for m in F32W_ROWS if m > 768]),
    ("NORM_F32W", 576, 192, [m for m in F32W_QKV_ROWS if m > 448])])
def test_row_lists_take_each_block_shape(form, n, k, rows):
    """The row counts of the tests below run every block shape of a form, in its store, SwiGLU,
    residual and qkv epilogues."""
    from mdlarc_scale_amd import _lib

    code = ["NORM", "SPLIT", "NORM_F32W", "SPLIT_F32W"].index(form)
    picks = {_lib.lib().mdl_prefill_gemm_pick(code, m, n, k) for m in rows}
    assert picks == set(range(_lib.lib().mdl_prefill_gemm_shapes(code)))


@pytest.mark.parametrize("k", [768, 1952, 1984])   # odd multiples of 32, past gamma's 1,920
def test_rows_do_not_depend_on_the_row_count(k):
    """Every block shape sums in the same order, so the first m rows of a product are the same bits
    whatever m is: each form at row counts that take each shape, against the rows of one large
    product (which the tests above pin to fp64)."""
    f, total = 2048, MANY_ROWS
    g = torch.Generator(DEV).manual_seed(k)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    wgu = K().tile_matrix((0.05 * rnd(2 * f, k)).to(torch.bfloat16))
    wo = K().tile_matrix((0.05 * rnd(768, k)).to(torch.bfloat16))
    x, gam, bias = rnd(total, k), 1 + 0.1 * rnd(k), rnd(f)
    a, res = torch.cat(split(rnd(total, k)), 1).contiguous(), rnd(total, 768)

    def forms(m):
        xt, at = K().tile_f32(x[:m]), K().tile_matrix(a[:m].contiguous())
        store, rs = torch.empty(m, 2 * f, device=DEV), torch.empty(m, device=DEV)
        K().prefill_gemm_norm(xt, gam, 1e-5, wgu, store, rs, k)
        h = torch.empty(K().split_numel(m, f, True), dtype=torch.bfloat16, device=DEV)
        K().prefill_gemm_norm_swiglu(xt, gam, 1e-5, wgu, bias, bias, h, m, f, k)
        out = torch.empty(m, 768, device=DEV)
        K().prefill_gemm_split(at, wo, out, k, a_tiled=True)
        xr = K().tile_f32(res[:m])
        K().prefill_gemm_split_residual(at, wo, xr, bias, m, 768, k, a_tiled=True)
        return store, rs, K().untile_matrix(h, m, 2 * f), out, K().untile_f32(xr, m, 768)

    whole = forms(total)
    for m in ROUTE_ROWS:
        for name, got, want in zip(("store", "rstd", "swiglu", "split", "residual"), forms(m),
                                   whole):
            assert torch.equal(got, want[:m]), f"{name} at {m} rows"


@pytest.mark.parametrize("m", ROUTE_ROWS + [MANY_QKV_ROWS])
def test_norm_qkv_at_each_block_shape(m):
    """The qkv epilogue of each shape against the E_STORE form and K2, bit for bit."""
    H, d = 12, 768
    g = torch.Generator(DEV).manual_seed(m)
    x = torch.randn(m, d, generator=g, device=DEV)
    gam = 1 + 0.1 * torch.randn(d, generator=g, device=DEV)
    w = K().tile_matrix((0.05 * torch.randn(3 * d, d, generator=g, device=DEV)).to(torch.bfloat16))
    pos = torch.randint(0, 35, (m, 3), generator=g, device=DEV)
    tab, geom = _rope()
    xt = K().tile_f32(x)
    qkv, rs1, rs2 = torch.empty(m, 3 * d, device=DEV), *torch.empty(2, m, device=DEV).unbind()
    K().prefill_gemm_norm(xt, gam, 1e-5, w, qkv, rs1, d)
    bf = lambda *s: torch.full(s, 7.0, dtype=torch.bfloat16, device=DEV)  # noqa: E731
    q1, kc1, vc1 = bf(m, d), bf(1, H, m + 3, 64), bf(1, H, m + 3, 64)
    K().qkv_rope_cache(qkv, rs1, pos, tab, geom, 1, m, H, 0.125, q1, kc1, vc1, slot0=0)
    q2, kc2, vc2 = bf(m, d), bf(1, H, m + 3, 64), bf(1, H, m + 3, 64)
    lead = torch.full((m, 3 * d), float("nan"), device=DEV)
    K().prefill_gemm_norm_qkv(xt, gam, 1e-5, w, m, H, rs2, lead, K().LEAD_QUERIES, None, pos, tab,
                              geom, 0.125, q2, kc2, vc2, seq=m)
    for got, want in ((rs2, rs1), (q2, q1), (kc2, kc1), (vc2, vc1), (lead[:64], qkv[:64])):
        assert torch.equal(got, want)


# under 8 k-steps, 8, and more; narrow outputs and inputs stay on K5 for up to 2,048 and 1,024 rows
@pytest.mark.parametrize("k,n", [(96, 768), (224, 768), (256, 768), (704, 256), (768, 768),
                                 (1952, 768), (2048, 768)])
def test_fp32_weight_forms(k, n):
    """The fp32-weight forms: a large product against fp64 of the products they form, a_hi w +
    a_lo w + a_hi w_lo (fp32 sums: 2e-6, as above), and every row count, on K5 (a few rows)
    and K6, at the edges of the tiles, the same bits as those rows of the large product."""
    f, total = 704, 20_000
    g = torch.Generator(DEV).manual_seed(k)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    wg, wo = 0.05 * rnd(2 * f, k), 0.05 * rnd(n, k)
    (wg_h, wg_l), (wo_h, wo_l) = split(wg), split(wo)
    tiles = [K().tile_matrix(t) for t in (wg_h, wg_l, wo_h, wo_l)]
    x, gam, bias, res = rnd(total, k), 1 + 0.1 * rnd(k), rnd(f), rnd(total, n)
    hi, lo = split(rnd(total, k))
    a = torch.cat([hi, lo], 1).contiguous()

    def forms(m):
        xt, at = K().tile_f32(x[:m]), K().tile_matrix(a[:m].contiguous())
        store, rs = torch.empty(m, 2 * f, device=DEV), torch.empty(m, device=DEV)
        K().prefill_gemm_norm_f32w(xt, gam, 1e-5, tiles[0], tiles[1], store, rs, k)
        h = torch.empty(K().split_numel(m, f, True), dtype=torch.bfloat16, device=DEV)
        K().prefill_gemm_norm_swiglu_f32w(xt, gam, 1e-5, tiles[0], tiles[1], bias, None, h, m, f,
                                          k)
        xr = K().tile_f32(res[:m])
        K().prefill_gemm_split_residual_f32w(at, tiles[2], tiles[3], xr, None, m, n, k)
        return store, rs, K().untile_matrix(h, m, 2 * f), K().untile_f32(xr, m, n)

    whole = forms(total)
    th, tl = split(x * gam)
    d = torch.Tensor.double
    acc = (d(th) + d(tl)) @ d(wg_h).T + d(th) @ d(wg_l).T
    assert rel(whole[0], acc) < 2e-6
    ref = d(res) + (d(hi) + d(lo)) @ d(wo_h).T + d(hi) @ d(wo_l).T
    assert rel(whole[3], ref) < 2e-6
    blocks = (acc / torch.sqrt((d(x) ** 2).mean(1, keepdim=True) + 1e-5)).view(total, -1, 2, 16)
    gate = blocks[:, :, 0].reshape(total, f) + d(bias)
    ref = torch.nn.functional.silu(gate) * blocks[:, :, 1].reshape(total, f)
    h = d(whole[2])
    assert rel(h[:, :f] + h[:, f:], ref) < 2e-5          # as the bf16 form's: the split of h
    for m in F32W_ROWS:
        for name, got, want in zip(("store", "rstd", "swiglu", "residual"), forms(m), whole):
            assert torch.equal(got, want[:m]), f"{name} at {m} rows"


def _f32w_qkv_inputs(m, H, seed):
    d = 64 * H
    g = torch.Generator(DEV).manual_seed(seed)
    wh, wl = split(0.05 * torch.randn(3 * d, d, generator=g, device=DEV))
    x = K().tile_f32(torch.randn(m, d, generator=g, device=DEV))
    gam = 1 + 0.1 * torch.randn(d, generator=g, device=DEV)
    pos = torch.randint(-2, 40, (m, 3), generator=g, device=DEV)   # clamped past the table's ends
    return x, gam, K().tile_matrix(wh), K().tile_matrix(wl), pos, *_rope()


@pytest.mark.parametrize("H", [3, 4, 12])
@pytest.mark.parametrize("m", F32W_QKV_ROWS)
@pytest.mark.parametrize("packed", [False, True])
def test_norm_qkv_of_fp32_weights(m, H, packed):
    """The fp32 qkv epilogue against the E_STORE form and K2, bit for bit; a packed list with
    tokens that have no slot, in a cache whose other slots stay as they were."""
    d = 64 * H
    x, gam, w, wl, pos, tab, geom = _f32w_qkv_inputs(m, H, m + H)
    qkv, rs = torch.empty(m, 3 * d, device=DEV), torch.empty(m, device=DEV)
    K().prefill_gemm_norm_f32w(x, gam, 1e-5, w, wl, qkv, rs, d)
    full = lambda *s: torch.full(s, 7.0, device=DEV)  # noqa: E731
    B, slots = (5, m + 3) if packed else (1, m + 3)
    want = full(m, d), full(B, H, slots, 64), full(B, H, slots, 64)
    got = full(m, d), full(B, H, slots, 64), full(B, H, slots, 64)
    scratch = torch.empty(m, 3 * d, device=DEV), torch.empty(m, device=DEV)
    if packed:
        row = torch.arange(m, device=DEV, dtype=torch.int32) * 5 // m
        slot = torch.arange(m, device=DEV, dtype=torch.int32) + 2
        slot[::7] = -1
        K().qkv_rope_cache_packed(qkv, rs, pos, tab, geom, row, slot, H, 0.125, *want)
        K().prefill_gemm_norm_qkv_f32w(x, gam, 1e-5, w, wl, m, H, *scratch, pos, tab, geom, 0.125,
                                       *got, token_row=row, token_slot=slot)
    else:
        K().qkv_rope_cache(qkv, rs, pos, tab, geom, 1, m, H, 0.125, *want, slot0=0)
        K().prefill_gemm_norm_qkv_f32w(x, gam, 1e-5, w, wl, m, H, *scratch, pos, tab, geom, 0.125,
                                       *got, seq=m)
    for name, a, b in zip("q K V".split(), got, want):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("m,H", [(1, 4), (16, 12), (17, 3), (250, 20)])
@pytest.mark.parametrize("t", [0, 5, 9])
def test_decode_norm_qkv_of_fp32_weights(m, H, t):
    """K5's fp32 qkv epilogue against gemm_norm and K2, bit for bit, in slot t of 10 alone."""
    d = 64 * H
    x, gam, w, wl, pos, tab, geom = _f32w_qkv_inputs(m, H, m + t)
    qkv, rs = torch.empty(m, 3 * d, device=DEV), torch.empty(m, device=DEV)
    slot = torch.tensor([t], dtype=torch.int32, device=DEV)
    for tile in range(0, 7):
        full = lambda *s: torch.full(s, 7.0, device=DEV)  # noqa: E731
        want = full(m, d), full(m, H, 10, 64), full(m, H, 10, 64)
        got = full(m, d), full(m, H, 10, 64), full(m, H, 10, 64)
        K().gemm_norm(x, gam, 1e-5, w, qkv, rs, d, tile=tile, w_lo=wl)
        K().qkv_rope_cache(qkv, rs, pos, tab, geom, m, 1, H, 0.125, *want, slot_dev=slot)
        K().gemm_norm_qkv(x, gam, 1e-5, w, m, H, None, pos, tab, geom, 0.125, *got,
                          slot_dev=slot, tile=tile, w_lo=wl)
        for name, a, b in zip("q K V".split(), got, want):
            assert torch.equal(a, b), f"{name} at tile {tile}"
