"""Several activation rows against one resident matrix on the matrix cores
(k3_skinny.hip): the spine projections, MXFP4 GEMVs and the one-expert launch
at the edges of their tiles, against a float64 reference.

Bounds.  Per element: a sum is rounded at most once for every eight of its
products (cols / 8 and 16 for its last steps), each time by 2^-24 of the sum of
|w x|; this is loose, and finds outputs that are wrong by themselves.  In norm: of
fp32 results the distance from float64 stays under 2^-21 of |w| |x| (rows and
positions together, growing with the root of the columns above 2,048): a sum of
random signs passes through some 30 to 60 roundings of 2^-24, about 2e-7, and what
is measured is 1e-7.  A lost third term of an activation costs 4e-6, ten times the
bound.  BF16 outputs are rounded by 2^-8 of the result once more.
"""
import pytest

pytestmark = pytest.mark.gpu

# rows around 16-row tiles and the row counts where 2 and 4 tiles start
ROWS = [1, 16, 17, 40, 4100, 8200]
POSITIONS = [1, 2, 3, 4, 5, 8, 9, 16, 17, 33, 64]


def _bound(w, x, cols, ref, bf16_out=False):
    b = (cols / 8 + 16) * 2.0 ** -24 * (x.abs() @ w.abs().t()) + 1e-30
    return b + 2.0 ** -8 * ref.abs() if bf16_out else b


def _check(out, w, x, cols, tag, bf16_out=False):
    ref = x @ w.t()
    err = (out.double() - ref).abs()
    bad = err > _bound(w, x, cols, ref, bf16_out)
    assert not bad.any(), f"{tag}: {int(bad.sum())} outputs off, worst {err.max().item():.3e}"
    if not bf16_out:
        norm = (err.norm() / (w.norm() * x.norm() + 1e-300)).item()
        assert norm <= 2.0 ** -21 * max(1.0, cols / 2048) ** 0.5, f"{tag}: {norm:.2e} of |w| |x|"


def _spine(kind, rows, cols, m, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, cols, generator=g, device="cuda")
    if kind == "bf16":
        w = torch.randn(rows, cols, generator=g, device="cuda").to(torch.bfloat16)
        return w, None, x, w.double()
    w = torch.randint(-128, 128, (rows, cols), generator=g, device="cuda", dtype=torch.int8)
    s = torch.rand(rows, generator=g, device="cuda") + 0.5
    return w, s, x, w.double() * s.double().unsqueeze(1)


def _run_spine(kind, w, s, x):
    from deltafin_amd import spine
    return spine.bf16_gemv(w, x) if kind == "bf16" else spine.int8_gemv(w, s, x)


@pytest.mark.parametrize("kind,cols", [("bf16", 32), ("bf16", 64), ("bf16", 72), ("bf16", 1000),
                                       ("bf16", 2048), ("int8", 64), ("int8", 144),
                                       ("int8", 1040), ("int8", 2048)])
def test_spine_edges(gpu, kind, cols):
    for i, rows in enumerate(ROWS):
        for m in POSITIONS if cols in (1000, 1040) else POSITIONS[i % 2::3]:
            print(f"[gpu-case] {kind} {rows}x{cols} positions {m}", flush=True)
            w, s, x, w64 = _spine(kind, rows, cols, m, rows + m)
            _check(_run_spine(kind, w, s, x), w64, x.double(), cols, f"{kind} {rows}x{cols} p{m}")


def _mxfp4(rows, cols, seed, lo=117, hi=121):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    p = torch.randint(0, 256, (rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = torch.randint(lo, hi + 1, (rows, cols // 32), generator=g, device="cuda",
                      dtype=torch.uint8)
    return p, s


def _dequant(p, s):
    import torch
    v = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]
    lut = torch.tensor(v + [-a for a in v], dtype=torch.float64, device="cuda")
    codes = torch.stack((p & 15, p >> 4), dim=-1).reshape(p.shape[0], -1).long()
    e = s.double()
    scale = torch.where(e == 0, 0.0, torch.exp2(e - 127.0))
    return lut[codes] * scale.repeat_interleave(32, dim=1)


@pytest.mark.parametrize("cols", [256, 288, 352, 1056, 2048])
@pytest.mark.parametrize("x_dtype", ["f32", "bf16"])
def test_mxfp4_edges(gpu, cols, x_dtype):
    import torch
    from deltafin_amd import moe
    for i, rows in enumerate(ROWS):
        p, s = _mxfp4(rows, cols, rows)
        w = _dequant(p, s)
        # scales at an odd address, which the interface allows
        odd = torch.empty(s.numel() + 1, dtype=torch.uint8, device="cuda")[1:]
        odd.copy_(s.reshape(-1))
        for m in (POSITIONS + [100])[i % 2::2]:
            print(f"[gpu-case] mxfp4 {rows}x{cols} {x_dtype} rows of x {m}", flush=True)
            x = torch.randn(m, cols, device="cuda").to(
                torch.float32 if x_dtype == "f32" else torch.bfloat16)
            for out in (torch.float32, torch.bfloat16):
                y = moe.mxfp4_gemv(p, odd, x, rows, cols, out_dtype=out)
                _check(y, w, x.double(), cols, f"mxfp4 {rows}x{cols} {x_dtype} m{m}",
                       out == torch.bfloat16)


def test_mxfp4_widest_row(gpu):
    """64 KB of activation is the widest row, whatever the number of rows."""
    import torch
    from deltafin_amd import _lib, moe
    for dt, cols in ((torch.float32, 16384), (torch.bfloat16, 32768)):
        for m in (1, 2, 5):
            x = torch.randn(m, cols, device="cuda").to(dt)
            p, s = _mxfp4(17, cols, m)
            _check(moe.mxfp4_gemv(p, s, x, 17, cols), _dequant(p, s), x.double(), cols, f"{dt} m{m}")
            p, s = _mxfp4(17, cols + 32, m)
            x = torch.randn(m, cols + 32, device="cuda").to(dt)
            with pytest.raises(_lib.K3HipError, match="too wide"):
                moe.mxfp4_gemv(p, s, x, 17, cols + 32)


@pytest.mark.parametrize("hidden,inter", [(256, 256), (3584, 3072), (1056, 352), (224, 64)])
def test_expert_rows(gpu, hidden, inter):
    """moe_launch at 1..17 rows (224 / 64: below a whole line, the separate launches)."""
    import torch
    from deltafin_amd import moe
    g = moe.geometry(hidden, inter, moe.K3_ACT_SITU)
    off = moe.span_offsets(g)
    span = torch.empty(off["span"], dtype=torch.uint8, device="cuda").random_(0, 256)
    mats = {}
    for name, a, b, c, r, k in (("gate", "w1p", "w1s", "w2p", inter, hidden),
                                ("down", "w2p", "w2s", "w3p", hidden, inter),
                                ("up", "w3p", "w3s", "span", inter, hidden)):
        span[off[b]:off[c]].random_(117, 122)
        mats[name] = _dequant(span[off[a]:off[b]].reshape(r, -1), span[off[b]:off[c]].reshape(r, -1))
    for m in (1, 2, 4, 7, 8, 16, 17):
        print(f"[gpu-case] expert {hidden}/{inter} rows {m}", flush=True)
        x = torch.randn(m, hidden, device="cuda")
        h, out = moe.moe_launch(g, span, x)
        gate, up = x.double() @ mats["gate"].t(), x.double() @ mats["up"].t()
        ref = 4 * torch.tanh(gate / 4) * torch.sigmoid(gate) * (25 * torch.tanh(up / 25))
        # the activation's slopes are at most 1.1 |up| and 4: the sums' bounds scaled by
        # them, and a few roundings of its own
        tol = (4.0 + 1.1 * up.abs()) * (_bound(mats["gate"], x.double(), hidden, gate)
                                        + _bound(mats["up"], x.double(), hidden, up)) \
            + 2.0 ** -20 * (ref.abs() + 1e-3)
        assert ((h.double() - ref).abs() <= tol).all(), f"h {hidden}/{inter} m{m}"
        _check(out, mats["down"], h.double(), inter, f"expert {hidden}/{inter} m{m}")


# |x| around 1, where the lower terms of an fp32 activation are subnormal in BF16
# (below 2^-110) and where x itself is subnormal
EXPONENTS = [0, -100, -112, -120, -126, -132]


@pytest.mark.parametrize("e", EXPONENTS)
def test_small_activations(gpu, e):
    """Activations of any size lose no bits: large weights bring every result to
    about 1, and the results' distance from 64 bits in norm stays at fp32's.  A
    sum is rounded once per matrix step or FMA, to 2^-24 of the partial sum; over
    the 64 steps of 2,048 columns such errors add to about 8 x 2^-24 / sqrt(3) =
    2.8e-7 of a sum of random signs.  4.8e-7 = 2^-21 is under twice that; a lost
    third term costs 4e-6."""
    import torch
    from deltafin_amd import moe
    rows, cols = 80, 2048
    scale = 2.0 ** min(100, -e)

    def near(y, ref, tag):
        err = ((y.double() - ref).norm() / ref.norm()).item()
        assert err <= 2.0 ** -21, f"{tag} at 2^{e}: {err:.2e}"

    for m in (2, 7, 16):
        print(f"[gpu-case] x at 2^{e}, {m} rows", flush=True)
        x0 = torch.randn(m, cols, device="cuda", dtype=torch.float64)
        x = (x0 * 2.0 ** e).float()
        w, _, _, _ = _spine("bf16", rows, cols, m, m)
        w = (w.float() * scale).to(torch.bfloat16)
        near(_run_spine("bf16", w, None, x), x.double() @ w.double().t(), "bf16")
        if e > -126:  # int8: the scale comes after the sum, which is subnormal below
            w, s, _, w64 = _spine("int8", rows, cols, m, m)
            near(_run_spine("int8", w, s * scale, x), x.double() @ (w64 * scale).t(), "int8")
        p, _ = _mxfp4(rows, cols, m)
        p &= 0xBB  # codes up to 1.5: exact in BF16 at every scale byte
        s = torch.full((rows, cols // 32), 127 + int(min(100, -e)), device="cuda",
                       dtype=torch.uint8)
        near(moe.mxfp4_gemv(p, s, x, rows, cols), x.double() @ _dequant(p, s).t(), "mxfp4")


def test_small_weights(gpu):
    """Weights that are subnormal in BF16 (E8M0 bytes 1 to 3 with codes of 0.5, BF16
    weights around 2^-130) count in full; byte 0 is +0."""
    import torch
    from deltafin_amd import moe
    rows, cols = 40, 2048
    for m in (2, 7, 16):
        print(f"[gpu-case] small weights, {m} rows", flush=True)
        x = torch.randn(m, cols, device="cuda") * 2.0 ** 100
        w = (torch.randn(rows, cols, device="cuda", dtype=torch.float64) * 2.0 ** -130).to(
            torch.bfloat16)
        cases = [("bf16", _run_spine("bf16", w, None, x), x, w.double())]
        p, _ = _mxfp4(rows, cols, m)
        p &= 0x99  # codes 0 and 0.5
        for byte in (0, 1, 2, 3):
            s = torch.full((rows, cols // 32), byte, device="cuda", dtype=torch.uint8)
            for v in (x, x.to(torch.bfloat16)):
                cases.append((f"byte {byte} {v.dtype}", moe.mxfp4_gemv(p, s, v, rows, cols), v,
                              _dequant(p, s)))
        for tag, y, v, w64 in cases:
            ref = v.double() @ w64.t()
            err = (y.double() - ref).norm().item()
            assert err <= 2.0 ** -21 * ref.norm().item(), f"{tag}, {m} rows: {err:.2e}"


def test_non_finite_inputs(gpu):
    """Infinities and NaN give what plain fp32 sums give: an infinite activation
    or weight its signed infinity, a NaN scale byte a NaN row, and a scale that
    overflows BF16 codes the finite result of its small products."""
    import torch
    from deltafin_amd import moe
    inf = float("inf")
    for kind in ("bf16", "int8"):
        w, s, x, w64 = _spine(kind, 40, 1040, 5, 3)
        x[1, 17] = inf
        x[2, 900] = -inf
        x[3, 5] = float("nan")
        # finite, where rounding it to BF16 would not be (int8: below the row scale's reach)
        x[4, 33] = 3.4028e38 if kind == "bf16" else 1e36
        if kind == "bf16":
            w[7, 100] = inf
            w64 = w.double()
        y = _run_spine(kind, w, s, x)
        ref = torch.stack([(x[i].double() * w64).sum(1) for i in range(5)])
        ref = torch.where(ref.abs() > 3.4028235e38, torch.sign(ref) * inf, ref)
        assert torch.equal(torch.isnan(y), torch.isnan(ref)), kind
        assert torch.equal(torch.isinf(y), torch.isinf(ref)), kind
        assert torch.equal(y[torch.isinf(y)].double(), ref[torch.isinf(ref)]), kind
        fin = torch.isfinite(ref)
        assert ((y.double() - ref)[fin].abs() <= 1e-4 * ref[fin].abs() + 1e-2).all(), kind
    p, s = _mxfp4(40, 512, 5)
    s[3, 7] = 255   # NaN row
    s[4, :] = 0     # zero row
    s[5, 2] = 254   # 2^127: codes above 2 overflow BF16
    p[5, 32:48] = 0x77  # all codes 6.0
    for dt in (torch.float32, torch.bfloat16):
        x = torch.randn(6, 512, device="cuda").to(dt)
        x[:, 64:96] = x[:, 64:96] * 2.0 ** -130
        w = _dequant(p, s)
        y = moe.mxfp4_gemv(p, s, x, 40, 512).double()
        assert torch.isnan(y[:, 3]).all() and not torch.isnan(y[:, [0, 1, 2, 4, 5, 6]]).any()
        assert (y[:, 4] == 0).all()
        ref = x.double() @ w.t()
        keep = [i for i in range(40) if i != 3]
        assert ((y - ref)[:, keep].abs() <= 1e-4 * (x.double().abs() @ w[keep].abs().t())).all()


@pytest.mark.parametrize("rows,m", [(33, 3), (40, 16), (4100, 16), (8200, 5), (4200, 33)])
@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp4"])
def test_non_finite_tiles(gpu, kind, rows, m):
    """Sums formed again at every place of a tile: each position but the last has an
    infinity, a NaN or a value whose scaled remainder overflows in some column; the
    outputs are those of float64, and the last position's stay what they are alone."""
    import torch
    from deltafin_amd import moe
    inf = float("inf")
    cols = 1056
    print(f"[gpu-case] non-finite {kind} {rows}x{cols} positions {m}", flush=True)
    if kind == "mxfp4":
        p, s = _mxfp4(rows, cols, rows + m)
        w64 = _dequant(p, s)
        x = torch.randn(m, cols, device="cuda")
        run = lambda x: moe.mxfp4_gemv(p, s, x, rows, cols)
    else:
        w, s, x, w64 = _spine(kind, rows, cols, m, rows + m)
        run = lambda x: _run_spine(kind, w, s, x)
    clean = x.clone()
    for i in range(m - 1):
        c = (7 + 131 * i) % cols
        x[i, c] = (inf, -inf, float("nan"), 2.0 ** 120 * (1.0 + 2.0 ** -7 - 2.0 ** -20))[i % 4]
    y, ref = run(x), x.double() @ w64.t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isinf(y), torch.isinf(ref))
    assert torch.equal(torch.sign(y[torch.isinf(y)]).double(), torch.sign(ref[torch.isinf(y)]))
    fin = torch.isfinite(ref)
    tol = 1e-5 * (torch.nan_to_num(x.double(), 0.0, 0.0, 0.0).abs() @ w64.abs().t())
    assert ((y.double() - ref).abs() <= tol)[fin].all()
    assert torch.equal(y[-1], run(clean)[-1])


def test_non_finite_cost(gpu):
    """A call whose every output is formed again stays within a small multiple of an
    ordinary one (one thread per output: 70 times; a wave per four: about 8)."""
    import torch
    for kind in ("bf16", "int8"):
        w, s, x, _ = _spine(kind, 7168, 6144, 16, 1)

        def us(x):
            for _ in range(3):
                _run_spine(kind, w, s, x)
            best = 1e9
            for _ in range(5):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                a.record()
                for _ in range(4):
                    _run_spine(kind, w, s, x)
                b.record()
                b.synchronize()
                best = min(best, a.elapsed_time(b) * 250)
            return best

        ordinary = us(x)
        x[:, 5000] = float("inf")
        again = us(x)
        print(f"[gpu-case] {kind}: {ordinary:.1f} us, formed again {again:.1f} us", flush=True)
        assert again <= 30 * ordinary, f"{kind}: {ordinary:.1f} us -> {again:.1f} us"
