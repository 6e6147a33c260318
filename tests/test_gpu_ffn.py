"""HIP grouped expert FFN forward/backward (MFMA kernels) against the CPU oracle, through the C ABI."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.util import rel_err, tol

pytestmark = pytest.mark.gpu


def _make(E, M, Fd, rows_per_expert, dtype, seed=0, pad_between=0):
    g = torch.Generator().manual_seed(seed)
    n = np.array(rows_per_expert, dtype=np.int32)
    off = np.zeros(E + 1, dtype=np.int32)
    off[1:] = np.cumsum(n + pad_between)
    R = int(off[-1])
    r = lambda *s, sc=1.0: (torch.randn(*s, generator=g) * sc).to(dtype)
    d = dict(xd=r(max(R, 1), M), w1=r(E, Fd, M, sc=0.05), b1=r(E, Fd, sc=0.05), w2=r(E, Fd, M, sc=0.05),
             b2=r(E, M, sc=0.05), go=r(max(R, 1), M), n=n, off=off, R=R)
    return d


def _oracle_fwd_bwd(d, gelu_bwd):
    """fp32 oracle on the same (rounded) inputs, per expert over its kept rows only."""
    f = {k: (v.float() if torch.is_tensor(v) else v) for k, v in d.items()}
    E = f["w1"].shape[0]
    R, M, Fd = d["R"], f["w1"].shape[2], f["w1"].shape[1]
    out = torch.zeros(max(R, 1), M); h = torch.zeros(max(R, 1), Fd)
    gx = torch.zeros(max(R, 1), M)
    g_w1 = torch.zeros_like(f["w1"]); g_w2 = torch.zeros_like(f["w2"])
    g_b1 = torch.zeros(E, Fd); g_b2 = torch.zeros(E, M)
    for e in range(E):
        lo, hi = int(d["off"][e]), int(d["off"][e]) + int(d["n"][e])
        if hi <= lo:
            continue
        o_e, h_e = O.ffn_fwd(f["xd"][lo:hi][None], f["w1"][e:e + 1], f["b1"][e:e + 1], f["w2"][e:e + 1], f["b2"][e:e + 1])
        out[lo:hi], h[lo:hi] = o_e[0], h_e[0]
        a, b, c_, dd, ee = O.ffn_bwd(f["go"][lo:hi][None], f["xd"][lo:hi][None], h_e, f["w1"][e:e + 1], f["w2"][e:e + 1], gelu_bwd)
        g_w1[e], g_b1[e], g_w2[e], g_b2[e], gx[lo:hi] = a[0], b[0], c_[0], dd[0], ee[0]
    return out, h, gx, g_w1, g_b1, g_w2, g_b2


CASES = [
    # E, M, F, rows per expert, gap between experts (padded layout has gaps)
    (1, 64, 128, [5], 0),
    (4, 64, 128, [130, 0, 7, 64], 0),
    (3, 136, 264, [257, 31, 129], 3),
    (8, 256, 512, [100, 200, 0, 1, 300, 128, 127, 129], 0),
    (2, 512, 2048, [1024, 1000], 24),
    # more experts than one wave of the tile search covers, most of them nearly empty
    (150, 64, 256, [(7 * e) % 23 if e % 3 else 0 for e in range(149)] + [700], 0),
    # an expert with more rows than four 320-row tiles, and column counts that are not whole tiles
    (3, 264, 520, [1500, 3, 321], 5),
    # more than 16 rounds of tiles (the grouped kernel then numbers them in plain expert order)
    (150, 64, 4096, [257 + (11 * e) % 90 for e in range(150)], 0),
    # experts of eight or more m-tiles (their tiles are numbered in groups of 8 n-tiles, the last group short: 9 and
    # 11 n-tiles here) beside experts that keep the plain order, one of them with a remainder tile of its own class
    (4, 64, 2304, [2100, 300, 0, 2600], 0),
    (3, 128, 2816, [2049, 1793, 2305], 8),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("gelu_bwd", ["tanh", "exact"])
@pytest.mark.parametrize("E,M,Fd,rows,gap", CASES)
def test_ffn_fwd_bwd_matches_oracle(E, M, Fd, rows, gap, gelu_bwd, dtype):
    from mole_amd import hip_ops as H, _lib as L
    print(f"ffn E={E} M={M} F={Fd} rows={rows} gap={gap} {gelu_bwd} {dtype}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=E * 7 + M, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    w_out, w_h, w_gx, w_gw1, w_gb1, w_gw2, w_gb2 = _oracle_fwd_bwd(d, gelu_bwd)
    t = tol(dtype)
    mask = torch.zeros(max(d["R"], 1), dtype=torch.bool)
    for e in range(E):
        mask[int(d["off"][e]):int(d["off"][e]) + int(d["n"][e])] = True
    assert rel_err(h.cpu()[mask], w_h[mask]) < t
    assert rel_err(out.cpu()[mask], w_out[mask]) < t
    assert rel_err(a.cpu()[mask], torch.nn.functional.gelu(w_h[mask])) < t
    g_w1 = torch.full_like(c["w1"], 9.0); g_w2 = torch.full_like(c["w2"], 9.0)
    g_b1 = torch.full_like(c["b1"], 9.0); g_b2 = torch.full_like(c["b2"], 9.0)
    mode = L.GELU_BWD_TANH if gelu_bwd == "tanh" else L.GELU_BWD_EXACT
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], g_w1, g_b1, g_w2, g_b2, True, False, mode)
    # the backward consumes the GPU's own saved h (rounded to the storage dtype), so compare against the
    # oracle evaluated on that same h for the tight fp32 bound
    assert rel_err(gx.cpu()[mask], w_gx[mask]) < t
    assert rel_err(g_w2, w_gw2) < t
    assert rel_err(g_b2, w_gb2) < t
    assert rel_err(g_w1, w_gw1) < t
    assert rel_err(g_b1, w_gb1) < t
    # accumulate variant (bffn_bwd_acc): a second call adds the same gradients again
    # (bf16: the running sum is rounded to bf16 after every call)
    H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], g_w1, g_b1, g_w2, g_b2, False, True, mode)
    assert rel_err(g_w1, 2 * w_gw1) < t and rel_err(g_b2, 2 * w_gb2) < t
    assert rel_err(g_w2, 2 * w_gw2) < t and rel_err(g_b1, 2 * w_gb1) < t


# The tile search: as many experts as a wave has lanes, one more, and more than the 256 whose rows a block holds; the last expert has rows, many
# have none, and an expert's last tile is full, above half a tile or below.  Every row against fp32 products of its own expert.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E", [64, 65, 257, 321])
def test_ffn_tiles_of_many_experts(E, dtype):
    from mole_amd import hip_ops as H
    print(f"ffn tiles of {E} experts {dtype}", flush=True)
    rows = [(0, 70, 128, 129, 200)[e % 5] for e in range(E - 1)] + [391]
    d = _make(E, 64, 136, rows, dtype, seed=E)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    out, h, a = H.ffn_fwd(c["xd"], torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda(), c["w1"], c["b1"], c["w2"], c["b2"])
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        if rows[e]:
            assert rel_err(h[r], c["xd"][r].float() @ c["w1"][e].float().t() + c["b1"][e].float()) < tol(dtype)
            assert rel_err(out[r], a[r].float() @ c["w2"][e].float() + c["b2"][e].float()) < tol(dtype)


# Backward products of many experts of few rows: contractions of one stage, of one and a rest, of three and of a rest and three.  (F = 1416 gives t more
# rows of tiles than 128 x 128 ones are taken for; the next test has the launches with rings of three stages.)
@pytest.mark.parametrize("M", [32, 40, 96, 104])
def test_ffn_backward_pair_with_three_stages(M):
    rows = [(30, 70, 128, 129, 1, 0, 100, 140)[e % 8] for e in range(32)]
    test_ffn_fwd_bwd_matches_oracle(32, M, 1416, rows, 0, "exact", torch.bfloat16)


# t and g_w2 in one launch with a ring of three stages (many tiles of few rows), results stored and added: contractions of one to four stages, which fill
# the ring and go round it, of one and a rest and of a rest and three; weight gradients of rows that end anywhere in a stage.
@pytest.mark.parametrize("M", [32, 40, 64, 96, 104, 128])
def test_ffn_backward_pair_on_the_ring_of_three_stages(M):
    from mole_amd import _lib as L
    rows = [(300, 70, 256, 129, 1, 0, 512, 652)[e % 8] for e in range(32)]
    assert [L.lib().mole_probe_pair_stages(32, sum(rows), M, 760, accumulate) for accumulate in (0, 1)] == [3, 3]
    test_ffn_fwd_bwd_matches_oracle(32, M, 760, rows, 0, "exact", torch.bfloat16)


# bf16 contractions that end inside a stage of 32 are summed in the order of k, those of whole stages as well: zeros behind them change no bit of h (K = M), out
# and gx (K = F).  One stage to eight, which every depth of a ring meets before and behind its end; tiles of 128 x 128 and of 256 columns, full and light ones.
@pytest.mark.parametrize("K", [8, 40, 72, 104, 136, 168, 200, 232])
@pytest.mark.parametrize("rows,N", [([130, 128, 70, 255, 100, 129, 200, 90] * 2, 512), ([1030, 1000, 700, 999, 1023, 900, 801, 1280] * 2, 1024)])
def test_ffn_zeros_behind_a_contraction_change_nothing(rows, N, K):
    from mole_amd import hip_ops as H, _lib as L
    print(f"zeros behind a contraction rows={sum(rows)} N={N} K={K}", flush=True)
    E, pad = 16, -K % 32
    def run(d, M, Fd):
        c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
        off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
        out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
        g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
        return h, out, H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g, True, False, L.GELU_BWD_TANH)
    behind = lambda t, dim: torch.cat([t, t.new_zeros(*[pad if i == dim % t.dim() else s for i, s in enumerate(t.shape)])], dim)
    d = _make(E, K, N, rows, torch.bfloat16, seed=K)
    wide = dict(d, **{k: behind(d[k], -1) for k in ("xd", "w1", "w2", "b2", "go")})
    assert torch.equal(run(d, K, N)[0], run(wide, K + pad, N)[0])
    d = _make(E, N, K, rows, torch.bfloat16, seed=K + 1)
    wide = dict(d, w1=behind(d["w1"], 1), w2=behind(d["w2"], 1), b1=behind(d["b1"], 1))
    for got, want in zip(run(d, N, K)[1:], run(wide, N, K + pad)[1:]):
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gemm_nt_gate_logits(dtype):
    from mole_amd import hip_ops as H
    print(f"gemm_nt {dtype}", flush=True)
    g = torch.Generator().manual_seed(1)
    for rows, N, K in [(1, 1, 8), (300, 16, 512), (1000, 256, 1024), (129, 100, 264)]:
        a = torch.randn(rows, K, generator=g).to(dtype); b = (torch.randn(N, K, generator=g) * 0.05).to(dtype)
        c = H.gemm_nt(a.cuda(), b.cuda())
        want = a.float() @ b.float().t()
        assert rel_err(c, want) < (1e-5 if dtype == torch.float32 else 1e-4)   # fp32 accumulation of exact products


@pytest.mark.parametrize("dtype,step", [(torch.bfloat16, 8), (torch.float32, 16), (torch.float32, 4)])
@pytest.mark.parametrize("seed", range(6))
def test_ffn_random_shapes(seed, dtype, step):
    """Random expert counts, loads and widths through the grouped kernels: 8-aligned widths for the bf16 direct-to-LDS
    kernel, 16-aligned ones for the fp32 one (whole stages of K), 4-aligned ones for the mix of the fp32 kernel (weight
    gradients) and the generic one (row-ragged products whose K is not whole stages)."""
    from mole_amd import hip_ops as H, _lib as L
    rng = np.random.default_rng(100 + seed)
    E = int(rng.integers(1, 40))
    M = int(rng.integers(1, 40)) * step
    Fd = int(rng.integers(1, 80)) * step
    rows = [int(r) for r in rng.choice([0, 1, 31, 32, 33, 63, 64, 65, 127, 129, 255, 256, 257, 320, 321, 640, 700], size=E)]
    gap = int(rng.integers(0, 3))
    print(f"ffn random seed={seed} {dtype} E={E} M={M} F={Fd} rows={rows} gap={gap}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=seed, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    w_out, w_h, w_gx, w_gw1, w_gb1, w_gw2, w_gb2 = _oracle_fwd_bwd(d, "tanh")
    t = tol(dtype)
    mask = torch.zeros(max(d["R"], 1), dtype=torch.bool)
    for e in range(E):
        mask[int(d["off"][e]):int(d["off"][e]) + int(d["n"][e])] = True
    if mask.any():
        assert rel_err(h.cpu()[mask], w_h[mask]) < t
        assert rel_err(out.cpu()[mask], w_out[mask]) < t
    g_w1 = torch.full_like(c["w1"], 9.0); g_w2 = torch.full_like(c["w2"], 9.0)
    g_b1 = torch.full_like(c["b1"], 9.0); g_b2 = torch.full_like(c["b2"], 9.0)
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], g_w1, g_b1, g_w2, g_b2, True, False, L.GELU_BWD_TANH)
    if mask.any():
        assert rel_err(gx.cpu()[mask], w_gx[mask]) < t
        assert rel_err(g_w2, w_gw2) < t and rel_err(g_b2, w_gb2) < t
        assert rel_err(g_w1, w_gw1) < t and rel_err(g_b1, w_gb1) < t
    else:   # no rows at all: every gradient is exactly zero
        for gt in (g_w1, g_b1, g_w2, g_b2):
            assert float(gt.float().abs().max()) == 0.0


def test_ffn_benchmark_size_against_fp32_products():
    """The benchmark's own shape (16 experts of 1024 -> 4096 -> 1024 in bf16, 16384 rows at uneven loads up to the
    capacity of 1280): forward and backward of three experts against fp32 torch products of the same rounded
    operands on the GPU (the CPU oracle would take minutes at this size), plus bias gradients of all experts."""
    from mole_amd import hip_ops as H, _lib as L
    E, M, Fd = 16, 1024, 4096
    g = torch.Generator().manual_seed(5)
    loads = torch.clamp((torch.randn(E, generator=g) * 120 + 1024).int(), min=1, max=1280)
    off = torch.zeros(E + 1, dtype=torch.int32)
    off[1:] = torch.cumsum(loads, 0)
    R = int(off[-1])
    print(f"ffn benchmark size: loads {loads.tolist()} R={R}", flush=True)
    dev, dt = "cuda", torch.bfloat16
    gd = torch.Generator(device=dev).manual_seed(6)
    rnd = lambda *s, sc=1.0: (torch.randn(*s, generator=gd, device=dev) * sc).to(dt)
    xd, go = rnd(R, M), rnd(R, M, sc=0.02)
    w1, b1, w2, b2 = rnd(E, Fd, M, sc=0.03), rnd(E, Fd, sc=0.03), rnd(E, Fd, M, sc=0.03), rnd(E, M, sc=0.03)
    offd, nd = off.cuda(), loads.int().cuda()
    out, h, a = H.ffn_fwd(xd, offd, nd, w1, b1, w2, b2)
    g_w1, g_b1, g_w2, g_b2 = torch.empty_like(w1), torch.empty_like(b1), torch.empty_like(w2), torch.empty_like(b2)
    gx = H.ffn_bwd(go, xd, h, a, offd, nd, w1, w2, g_w1, g_b1, g_w2, g_b2, True, False, L.GELU_BWD_EXACT)
    torch.cuda.synchronize()
    t = tol(dt)
    for e in (0, 7, 15):
        lo, hi = int(off[e]), int(off[e + 1])
        x32, go32 = xd[lo:hi].float(), go[lo:hi].float()
        h32 = x32 @ w1[e].float().t() + b1[e].float()
        a32 = torch.nn.functional.gelu(h32)
        o32 = a32 @ w2[e].float() + b2[e].float()
        assert rel_err(h[lo:hi], h32) < t and rel_err(a[lo:hi], a32) < t and rel_err(out[lo:hi], o32) < t
        # backward from the kernel's own (bf16) h, as the kernel sees it
        hs = h[lo:hi].float()
        hs.requires_grad_(True)
        torch.nn.functional.gelu(hs).backward(go32 @ w2[e].float().t())
        t32 = hs.grad
        assert rel_err(g_w2[e], a[lo:hi].float().t() @ go32) < t
        assert rel_err(g_w1[e], t32.t() @ x32) < t
        assert rel_err(gx[lo:hi], t32 @ w1[e].float()) < t
        assert rel_err(g_b1[e], t32.sum(0)) < t
    # bias gradient of the second linear for every expert: plain column sums of go
    want_b2 = torch.stack([go[int(off[e]):int(off[e + 1])].float().sum(0) for e in range(E)])
    assert rel_err(g_b2, want_b2) < t


def test_ffn_imbalanced_full_size_against_fp32_products():
    """The imbalanced configuration at its real shape (64 experts of 2048 -> 8192 -> 2048 in bf16, 16384 kept rows,
    expert loads from a Zipf-biased top-2 routing: a handful of rows up to well over a thousand): the lightest, a
    middle and the heaviest expert against fp32 torch products of the same rounded operands, forward and backward."""
    from mole_amd import hip_ops as H, _lib as L
    from tests.util import zipf_scores
    S, E, k, M, Fd = 8192, 64, 2, 2048, 8192
    r = H.route(zipf_scores(S, E, seed=11).cuda(), k, 0.0)
    loads = r.kept_rows.cpu()
    off = r.offsets.cpu()
    R = int(off[-1])
    assert R == S * k
    order = torch.argsort(loads)
    picks = [int(order[0]), int(order[E // 2]), int(order[-1])]
    print(f"ffn imbalanced full size: loads min {int(loads.min())} median {int(loads.median())} max {int(loads.max())}, "
          f"experts {picks}", flush=True)
    dev, dt = "cuda", torch.bfloat16
    gd = torch.Generator(device=dev).manual_seed(12)
    rnd = lambda *s, sc=1.0: (torch.randn(*s, generator=gd, device=dev) * sc).to(dt)
    xd, go = rnd(R, M), rnd(R, M, sc=0.02)
    w1, b1, w2, b2 = rnd(E, Fd, M, sc=0.02), rnd(E, Fd, sc=0.02), rnd(E, Fd, M, sc=0.02), rnd(E, M, sc=0.02)
    out, h, a = H.ffn_fwd(xd, r.offsets, r.kept_rows, w1, b1, w2, b2)
    g_w1, g_b1, g_w2, g_b2 = torch.empty_like(w1), torch.empty_like(b1), torch.empty_like(w2), torch.empty_like(b2)
    gx = H.ffn_bwd(go, xd, h, a, r.offsets, r.kept_rows, w1, w2, g_w1, g_b1, g_w2, g_b2, True, False, L.GELU_BWD_TANH)
    torch.cuda.synchronize()
    t = tol(dt)
    c = 0.7978845608028654
    for e in picks:
        lo, hi = int(off[e]), int(off[e + 1])
        if hi == lo:
            assert float(g_w1[e].float().abs().max()) == 0.0 and float(g_w2[e].float().abs().max()) == 0.0
            continue
        x32, go32 = xd[lo:hi].float(), go[lo:hi].float()
        h32 = x32 @ w1[e].float().t() + b1[e].float()
        assert rel_err(h[lo:hi], h32) < t
        assert rel_err(a[lo:hi], torch.nn.functional.gelu(h32)) < t
        assert rel_err(out[lo:hi], torch.nn.functional.gelu(h32) @ w2[e].float() + b2[e].float()) < t
        hs = h[lo:hi].float()                      # the derivative the reference compiles (MOLE/cpp/gelu.cu:3-14)
        th = torch.tanh(c * (hs + 0.044715 * hs ** 3))
        dg = 0.5 * (1 + th) + 0.5 * hs * c * (1 - th * th) * (1 + 3 * 0.044715 * hs * hs)
        t32 = (go32 @ w2[e].float().t()) * dg
        assert rel_err(g_w2[e], a[lo:hi].float().t() @ go32) < t
        assert rel_err(g_w1[e], t32.t() @ x32) < t
        assert rel_err(gx[lo:hi], t32 @ w1[e].float()) < t
        assert rel_err(g_b1[e], t32.sum(0)) < t
        assert rel_err(g_b2[e], go32.sum(0)) < t


def test_ffn_fine_grained_full_size_against_fp32_products():
    """The fine-grained configuration at its real shape (256 experts of 2048 -> 1024 -> 2048 in bf16, top-8 of
    32768 tokens: 262144 kept rows, about a thousand per expert, more than 16 rounds of tiles per launch): three
    experts against fp32 torch products of the same rounded operands, forward and backward (exact GELU')."""
    from mole_amd import hip_ops as H, _lib as L
    S, E, k, M, Fd = 32768, 256, 8, 2048, 1024
    dev, dt = "cuda", torch.bfloat16
    gd = torch.Generator(device=dev).manual_seed(21)
    scores = torch.softmax(torch.randn(S, E, generator=gd, device=dev), -1)
    r = H.route(scores, k, 0.0)
    off = r.offsets.cpu()
    R = int(off[-1])
    assert R == S * k
    print(f"ffn fine-grained full size: loads {int(r.kept_rows.min())}..{int(r.kept_rows.max())}", flush=True)
    rnd = lambda *s, sc=1.0: (torch.randn(*s, generator=gd, device=dev) * sc).to(dt)
    xd, go = rnd(R, M), rnd(R, M, sc=0.02)
    w1, b1, w2, b2 = rnd(E, Fd, M, sc=0.02), rnd(E, Fd, sc=0.02), rnd(E, Fd, M, sc=0.02), rnd(E, M, sc=0.02)
    out, h, a = H.ffn_fwd(xd, r.offsets, r.kept_rows, w1, b1, w2, b2)
    g_w1, g_b1, g_w2, g_b2 = torch.empty_like(w1), torch.empty_like(b1), torch.empty_like(w2), torch.empty_like(b2)
    gx = H.ffn_bwd(go, xd, h, a, r.offsets, r.kept_rows, w1, w2, g_w1, g_b1, g_w2, g_b2, True, False, L.GELU_BWD_EXACT)
    torch.cuda.synchronize()
    t = tol(dt)
    for e in (0, 131, 255):
        lo, hi = int(off[e]), int(off[e + 1])
        x32, go32 = xd[lo:hi].float(), go[lo:hi].float()
        h32 = x32 @ w1[e].float().t() + b1[e].float()
        assert rel_err(h[lo:hi], h32) < t
        assert rel_err(out[lo:hi], torch.nn.functional.gelu(h32) @ w2[e].float() + b2[e].float()) < t
        hs = h[lo:hi].float()
        hs.requires_grad_(True)
        torch.nn.functional.gelu(hs).backward(go32 @ w2[e].float().t())
        t32 = hs.grad
        assert rel_err(g_w2[e], a[lo:hi].float().t() @ go32) < t
        assert rel_err(g_w1[e], t32.t() @ x32) < t
        assert rel_err(gx[lo:hi], t32 @ w1[e].float()) < t
        assert rel_err(g_b1[e], t32.sum(0)) < t
        assert rel_err(g_b2[e], go32.sum(0)) < t


def _bf16_grid(limit=8.0, min_exp=-14):
    """Every bf16 value v with 2^min_exp <= |v| <= limit, and zero."""
    bits = torch.arange(0, 1 << 15, dtype=torch.int32)
    v = (bits << 16).view(torch.float32)
    v = v[torch.isfinite(v) & (v <= limit) & (v >= 2.0 ** min_exp)]
    return torch.cat([torch.zeros(1), v, -v])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_fused_activation_math_on_a_dense_grid(dtype):
    """The GELU of the forward epilogue and both GELU derivatives of the backward epilogue, pinned through the
    FFN entry points themselves on every bf16 value of magnitude 2^-14 .. 8 (about 4400 points): one-hot rows in
    w1 make h an exact copy of xd, one-hot rows in w2 make go . w2^T exactly 1, so a = gelu(h) and t = gelu'(h)
    rounded once to the buffer dtype.  bf16 results come from polynomial fits (stated absolute error 6e-5 for the
    GELU's erf part, 2e-4 for the derivatives); the bound is that error plus the rounding of the result (half a
    unit in the last place of its binade).  fp32 results come from the closed forms and are held to 2e-6."""
    from mole_amd import hip_ops as H, _lib as L
    grid = _bf16_grid()
    M, Fd = 64, 256
    rows = (grid.numel() + M - 1) // M
    vals = torch.zeros(rows * M)
    vals[:grid.numel()] = grid
    xd = vals.view(rows, M).to(dtype).cuda()
    w1 = torch.zeros(1, Fd, M)
    w1[0, torch.arange(Fd), torch.arange(Fd) % M] = 1.0          # h[r, f] = xd[r, f mod M]
    w2 = torch.zeros(1, Fd, M)
    w2[0, :, 0] = 1.0                                             # (go . w2^T)[r, f] = go[r, 0]
    b1, b2 = torch.zeros(1, Fd), torch.zeros(1, M)
    go = torch.zeros(rows, M)
    go[:, 0] = 1.0
    off = torch.tensor([0, rows], dtype=torch.int32).cuda()
    n = torch.tensor([rows], dtype=torch.int32).cuda()
    dev = lambda t: t.to(dtype).cuda()
    w1d, w2d = dev(w1), dev(w2)
    out, h, a = H.ffn_fwd(xd, off, n, w1d, dev(b1), w2d, dev(b2))
    h64 = xd.double().cpu().repeat(1, Fd // M)
    assert torch.equal(h.double().cpu(), h64)                     # the set-up: h is xd, exactly
    gelu64 = 0.5 * h64 * (1.0 + torch.erf(h64 / 2.0 ** 0.5))
    bits = 8 if dtype == torch.bfloat16 else 24          # significand bits of the buffer dtype

    def half_ulp(v, slack):
        """Half a unit in the last place of the binade that |v| + slack falls into (the result is rounded once)."""
        mag = torch.clamp(v.abs() + slack, min=2.0 ** -126)
        return torch.pow(2.0, torch.floor(torch.log2(mag)) - bits)

    poly = 6e-5 if dtype == torch.bfloat16 else 2e-6
    err = (a.double().cpu() - gelu64).abs()
    slack = poly * torch.clamp(h64.abs(), min=1.0)
    bound = slack + half_ulp(gelu64, slack)
    worst = float((err - half_ulp(gelu64, slack)).max())
    print(f"fused GELU {dtype}: worst error beyond rounding {worst:.2e}", flush=True)
    assert bool((err <= bound).all()), f"GELU off by {float((err / bound).max()):.2f}x its bound"
    for variant, fn, code in (("tanh", O.d_gelu_tanh, L.GELU_BWD_TANH), ("exact", O.d_gelu_exact, L.GELU_BWD_EXACT)):
        g_w1, g_b1, g_w2, g_b2 = (torch.empty_like(t) for t in (w1d, dev(b1), w2d, dev(b2)))
        t = torch.empty(rows, Fd, dtype=dtype, device="cuda")
        H.ffn_bwd_into(dev(go), xd, h, a, off, n, 1, rows, M, Fd, w1d, w2d, t, g_w1, g_b1, g_w2, g_b2, None, False, code)
        d64 = fn(h64)
        err = (t.double().cpu() - d64).abs()
        polyd = 2e-4 if dtype == torch.bfloat16 else 2e-6
        slack = torch.full_like(d64, polyd)
        bound = slack + half_ulp(d64, slack)
        worst = float((err - half_ulp(d64, slack)).max())
        print(f"fused GELU' ({variant}) {dtype}: worst error beyond rounding {worst:.2e}", flush=True)
        assert bool((err <= bound).all()), f"GELU' ({variant}) off by {float((err / bound).max()):.2f}x its bound"


# Experts of few rows: the streamed-weight kernels.  Rows around their 16-row blocks and 32-row groups, widths that end
# inside a step of the contraction, a 64- or 128-column tile, and contractions short and long enough to be split over
# blocks or not.  The tolerance is the one of every FFN test (fp32 sums of bf16 / fp32 products in another order).
FEW_ROWS = [
    (1, 64, 128, [1], 0),
    (4, 520, 1416, [1, 0, 15, 16], 0),
    (5, 136, 2056, [17, 1, 0, 31, 3], 2),
    (3, 264, 4096, [33, 16, 5], 1),
    (6, 1032, 520, [0, 2, 40, 1, 0, 64], 0),
    (70, 64, 1032, [(5 * e) % 9 for e in range(70)], 0),
    # where bf16's K-strided products change to tiles: below and from 32 and 48 tiles, at 24 / 12 rows an expert and one more;
    # without a workspace, where the tiles could not split the contraction, they stay
    (31, 64, 1032, [25 + e % 3 for e in range(31)], 0), (32, 64, 1032, [24 + (e % 3 - 1) for e in range(32)], 0),
    (32, 64, 1032, [25] * 32, 1), (48, 64, 1032, [12] * 48, 0), (48, 72, 1032, [13 + 4 * (e % 3 - 1) for e in range(48)], 0),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,M,Fd,rows,gap", FEW_ROWS)
def test_ffn_few_rows_matches_oracle(E, M, Fd, rows, gap, dtype):
    from mole_amd import hip_ops as H, _lib as L
    print(f"ffn few rows E={E} M={M} F={Fd} rows={rows} gap={gap} {dtype}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=E + M + Fd, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    w_out, w_h, w_gx, w_gw1, w_gb1, w_gw2, w_gb2 = _oracle_fwd_bwd(d, "tanh")
    mask = torch.zeros(max(d["R"], 1), dtype=torch.bool)
    for e in range(E):
        mask[int(d["off"][e]):int(d["off"][e]) + int(d["n"][e])] = True
    t = tol(dtype)
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.full_like(c[k], 9.0) for k in ("w1", "b1", "w2", "b2")]
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    for got, want in ((h, w_h), (a, torch.nn.functional.gelu(w_h)), (out, w_out), (gx, w_gx)):
        assert rel_err(got.cpu()[mask], want[mask]) < t
    for got, want in zip(g, (w_gw1, w_gb1, w_gw2, w_gb2)):
        assert rel_err(got, want) < t
    # without a workspace the contraction is not split over blocks: the same result to rounding
    out2, h2, a2 = torch.empty_like(out), torch.empty_like(h), torch.empty_like(a)
    L.check(L.lib().mole_ffn_fwd(L.ptr(c["xd"]), L.dtype_code(dtype), L.ptr(off), L.ptr(n), E, d["R"], M, Fd, L.ptr(c["w1"]),
                                 L.ptr(c["b1"]), L.ptr(c["w2"]), L.ptr(c["b2"]), L.ptr(h2), L.ptr(a2), L.ptr(out2), L.stream()), "ffn")
    assert torch.equal(h2.cpu()[mask], h.cpu()[mask]) and rel_err(out2.cpu()[mask], w_out[mask]) < t


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ffn_few_rows_leaves_other_experts_rows_alone(dtype):
    """A launch over some of the experts (offloaded experts run in chunks) with its contraction split over blocks: rows of
    experts outside the launch keep what they hold, in the forward's out and in the backward's gx."""
    from mole_amd import hip_ops as H
    E, M, Fd, rows = 4, 256, 4096, [3, 5, 2, 6]
    print(f"ffn few rows, chunk {dtype}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=3)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    R = d["R"]
    h, a = (torch.empty(R, Fd, dtype=dtype, device="cuda") for _ in range(2))
    t = torch.empty_like(h)
    out, gx = (torch.full((R, M), 7.0, dtype=dtype, device="cuda") for _ in range(2))
    w_out, _, w_gx, *_ = _oracle_fwd_bwd(d, "tanh")
    junk = torch.full((64 * R * M,), float("nan"), device="cuda")      # what the workspace's memory may hold
    del junk
    lo, hi = int(d["off"][1]), int(d["off"][3])
    ws = [c[k][1:3] for k in ("w1", "b1", "w2", "b2")]
    H.ffn_fwd_into(c["xd"], off[1:], n[1:], 2, R, M, Fd, *ws, h, a, out)
    g = [torch.empty_like(w) for w in ws]
    H.ffn_bwd_into(c["go"], c["xd"], h, a, off[1:], n[1:], 2, R, M, Fd, ws[0], ws[2], t, *g, gx, False, 0)
    assert rel_err(out.cpu()[lo:hi], w_out[lo:hi]) < tol(dtype) and rel_err(gx.cpu()[lo:hi], w_gx[lo:hi]) < tol(dtype)
    for buf in (out, gx):
        assert float((torch.cat([buf[:lo], buf[hi:]]) - 7.0).abs().max()) == 0.0


# bf16 contractions that end inside a 32-wide stage of the direct-to-LDS kernel: one short stage only, every remainder of 8,
# one and several stages before it; 128-row, 256-row and 320-row tiles (few experts, many rows, many experts).
@pytest.mark.parametrize("E,M,Fd,rows,gap", [
    (2, 8, 24, [300, 70], 0), (3, 40, 72, [129, 200, 31], 1), (2, 136, 520, [600, 257], 0), (4, 104, 1112, [90, 128, 0, 65], 0),
    (30, 264, 2088, [60 + (37 * e) % 90 for e in range(30)], 0), (40, 72, 1048, [300 + (29 * e) % 100 for e in range(40)], 0),
])
def test_ffn_contraction_ends_inside_a_stage(E, M, Fd, rows, gap):
    from mole_amd import hip_ops as H
    dtype = torch.bfloat16
    print(f"ffn K tail E={E} M={M} F={Fd} rows={rows[:4]}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=M + Fd, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    w_out, w_h, w_gx, *w_g = _oracle_fwd_bwd(d, "tanh")
    mask = torch.zeros(d["R"], dtype=torch.bool)
    for e in range(E):
        mask[int(d["off"][e]):int(d["off"][e]) + int(d["n"][e])] = True
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.full_like(c[k], 9.0) for k in ("w1", "b1", "w2", "b2")]
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    for got, want in ((h, w_h), (out, w_out), (gx, w_gx)):
        assert rel_err(got.cpu()[mask], want[mask]) < tol(dtype)
    for got, want in zip(g, w_g):
        assert rel_err(got, want) < tol(dtype)


# What whole stages of 32 leave of a contraction comes first: every such rest, alone, before one stage, two, and more than the ring holds.  Small
# whole numbers, whose sums are exact in any order: the results are the nearest bf16 numbers.
@pytest.mark.parametrize("E,M,Fd,rows,tile", [
    (6, 520, 264, [65, 71, 95, 96, 97, 127], 128), (5, 136, 256, [129, 159, 161, 191, 223], 128), (64, 512, 1024, [65 + (31 * e) % 260 for e in range(64)], 256)])
def test_ffn_contraction_with_its_rest_first(E, M, Fd, rows, tile):
    from mole_amd import hip_ops as H, _lib as L
    print(f"ffn rest first E={E} M={M} F={Fd} rows={rows[:6]}", flush=True)
    g = torch.Generator().manual_seed(E + M)
    whole = lambda *s: torch.randint(-3, 4, s, generator=g).bfloat16().cuda()
    off = torch.tensor([0] + list(np.cumsum(rows)), dtype=torch.int32).cuda(); n = torch.tensor(rows, dtype=torch.int32).cuda()
    R = sum(rows)
    assert L.lib().mole_probe_wgrad_tile(E, R, Fd, M) == tile
    a, go = whole(R, Fd), whole(R, M)
    w = whole(E, Fd, M)
    t = torch.zeros(R, Fd, dtype=torch.bfloat16, device="cuda")
    grads = [torch.full_like(q, 9.0) for q in (w, w[:, :, 0].contiguous(), w, w[:, 0].contiguous())]
    H.ffn_bwd_into(go, whole(R, M), a, a, off, n, E, R, M, Fd, w, w, t, *grads, None, False, L.GELU_BWD_EXACT)
    o = np.cumsum([0] + rows)
    for e in range(E):
        want = a[o[e]:o[e + 1]].double().t() @ go[o[e]:o[e + 1]].double()
        assert torch.equal(grads[2][e], want.bfloat16()) and torch.equal(grads[3][e], go[o[e]:o[e + 1]].double().sum(0).bfloat16())
    for K in (8, 40, 64, 72, 136, 248):
        p, q = whole(300, K), whole(72, K)
        want = p.double() @ q.double().t()
        assert torch.equal(H.gemm_nt(p, q).double(), want)
        assert torch.equal(H.gemm_nn(p, q.t().contiguous()), want.bfloat16())


# K = F products whose contraction is split into planes: 256- and 320-row tiles in two to four planes, 128 x 128 tiles in two to
# four, planes of unequal and of ragged length, columns that are not whole tiles, an expert with no rows; the two results
# with a workspace (split) and without one.
@pytest.mark.parametrize("E,M,Fd,rows,gap", [
    (3, 264, 3080, [330, 0, 200], 2), (4, 1032, 3104, [375, 370, 380, 20], 0), (30, 520, 2056, [100 + (7 * e) % 50 for e in range(30)], 0),
    (4, 72, 2088, [200, 130, 90, 300], 1), (2, 520, 1064, [129, 250], 0),
])
def test_ffn_split_contraction(E, M, Fd, rows, gap):
    from mole_amd import hip_ops as H, _lib as L
    dtype = torch.bfloat16
    print(f"ffn planes E={E} M={M} F={Fd} rows={rows[:4]}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=M + Fd, pad_between=gap)
    assert L.lib().mole_ffn_workspace_bytes(L.dtype_code(dtype), E, d["R"], M, Fd) > 0
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    w_out, _, w_gx, *_ = _oracle_fwd_bwd(d, "tanh")
    mask = torch.zeros(d["R"], dtype=torch.bool)
    for e in range(E):
        mask[int(d["off"][e]):int(d["off"][e]) + int(d["n"][e])] = True
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    assert rel_err(out.cpu()[mask], w_out[mask]) < tol(dtype) and rel_err(gx.cpu()[mask], w_gx[mask]) < tol(dtype)
    out2, h2, a2 = torch.empty_like(out), torch.empty_like(h), torch.empty_like(a)
    L.check(L.lib().mole_ffn_fwd(L.ptr(c["xd"]), L.dtype_code(dtype), L.ptr(off), L.ptr(n), E, d["R"], M, Fd, L.ptr(c["w1"]),
                                 L.ptr(c["b1"]), L.ptr(c["w2"]), L.ptr(c["b2"]), L.ptr(h2), L.ptr(a2), L.ptr(out2), L.stream()), "ffn")
    assert rel_err(out2.cpu()[mask], w_out[mask]) < tol(dtype)


# The same in fp32: 64 x 128 tiles in two to four planes of equal and of unequal length, columns that are not whole tiles,
# an expert with no rows, gaps between the experts.  Without a workspace the same products run in one piece; sums of the
# same fp32 terms in another order differ by a few rounding errors of the partial sums, far inside the tolerance.
@pytest.mark.parametrize("E,M,Fd,rows,gap", [
    (1, 132, 2064, [70], 0), (8, 512, 2048, [190 + e for e in range(8)], 2), (3, 68, 1040, [100, 0, 129], 1), (5, 260, 784, [65, 80, 193, 64, 90], 0),
])
def test_ffn_split_contraction_fp32(E, M, Fd, rows, gap):
    from mole_amd import hip_ops as H, _lib as L
    dtype = torch.float32
    print(f"ffn fp32 planes E={E} M={M} F={Fd} rows={rows[:4]}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=M + Fd, pad_between=gap)
    assert L.lib().mole_ffn_workspace_bytes(L.dtype_code(dtype), E, d["R"], M, Fd) > 0
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    w_out, _, w_gx, *_ = _oracle_fwd_bwd(d, "tanh")
    mask = torch.zeros(d["R"], dtype=torch.bool)
    for e in range(E):
        mask[int(d["off"][e]):int(d["off"][e]) + int(d["n"][e])] = True
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    assert rel_err(out.cpu()[mask], w_out[mask]) < tol(dtype) and rel_err(gx.cpu()[mask], w_gx[mask]) < tol(dtype)
    out2, h2, a2 = torch.empty_like(out), torch.empty_like(h), torch.empty_like(a)
    L.check(L.lib().mole_ffn_fwd(L.ptr(c["xd"]), L.dtype_code(dtype), L.ptr(off), L.ptr(n), E, d["R"], M, Fd, L.ptr(c["w1"]),
                                 L.ptr(c["b1"]), L.ptr(c["w2"]), L.ptr(c["b2"]), L.ptr(h2), L.ptr(a2), L.ptr(out2), L.stream()), "ffn")
    assert torch.equal(h2.cpu()[mask], h.cpu()[mask]) and rel_err(out2.cpu()[mask], w_out[mask]) < tol(dtype)


# bf16 weight gradients by 128 x 128 tiles: widths below, at and just past a tile's edge, contractions of less than one
# stage up to several rings of stages, experts without rows, written and added to what is there.
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("E,M,Fd,rows,gap", [
    (1, 8, 8, [1], 0), (3, 128, 128, [31, 0, 33], 0), (2, 136, 264, [64, 250], 1), (5, 520, 1416, [128, 97, 1, 0, 161], 2), (33, 72, 120, [(13 * e) % 70 for e in range(33)], 0),
])
def test_ffn_weight_gradients_by_small_tiles(E, M, Fd, rows, gap, accumulate):
    from mole_amd import hip_ops as H
    dtype = torch.bfloat16
    print(f"ffn weight gradients E={E} M={M} F={Fd} rows={rows[:5]} accumulate={accumulate}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=E + M + Fd, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    *_, w_gw1, w_gb1, w_gw2, w_gb2 = _oracle_fwd_bwd(d, "tanh")
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.full_like(c[k], 0.5) for k in ("w1", "b1", "w2", "b2")]
    H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g, accumulate=accumulate)
    for got, want in zip(g, (w_gw1, w_gb1, w_gw2, w_gb2)):
        assert rel_err(got, want + 0.5 if accumulate else want) < tol(dtype)


# Layers whose backward products all take 128 x 128 tiles run them in two launches, each a row-ragged product beside a weight gradient.
# A result in the place of an operand of the other product (t in a's place, gx in xd's) is not such a pair: the same launches one
# after the other give the same bits.  Whole stages and contractions that end inside one; planes; empty and skewed experts.
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("E,M,Fd,rows,gap", [
    (16, 520, 1416, [128, 97, 131, 0, 161] + [120] * 11, 0), (4, 512, 1024, [257, 228, 0, 255], 3), (2, 256, 1536, [200, 130], 0),
    (1, 136, 1032, [700], 0), (9, 320, 640, [30, 1, 400, 33, 64, 0, 65, 128, 129], 1)])
def test_ffn_backward_products_in_pairs(E, M, Fd, rows, gap, accumulate):
    from mole_amd import hip_ops as H, _lib as L
    print(f"ffn pairs E={E} M={M} F={Fd} accumulate={accumulate}", flush=True)
    d = _make(E, M, Fd, rows, torch.bfloat16, seed=E + M, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    R = d["R"]
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    ws = torch.empty(max(1, L.lib().mole_ffn_workspace_bytes(L.MOLE_BF16, E, R, M, Fd)), dtype=torch.uint8, device="cuda")
    res = []
    for in_place in (False, True):
        xd, a_ = c["xd"].clone(), a.clone()
        t = a_ if in_place else torch.zeros_like(a)
        gx = xd if in_place else torch.zeros_like(xd)
        g = [torch.full_like(c[k], 0.5) for k in ("w1", "b1", "w2", "b2")]
        L.kernel_timing_enable(True)
        L.kernel_timing_read()
        L.check(L.lib().mole_ffn_bwd_ws(L.ptr(c["go"]), L.ptr(xd), L.ptr(h), L.ptr(a_), L.MOLE_BF16, L.ptr(off), L.ptr(n), E, R, M, Fd, L.ptr(c["w1"]),
                                        L.ptr(c["w2"]), L.ptr(t), *[L.ptr(q) for q in g], L.ptr(gx), int(accumulate), L.GELU_BWD_TANH, L.ptr(ws), ws.numel(),
                                        L.stream()), "mole_ffn_bwd_ws")
        torch.cuda.synchronize()
        launches = {k: v[0] for k, v in L.kernel_timing_read().items() if k in ("ffn_gw1", "ffn_gw2")}
        L.kernel_timing_enable(False)
        assert sum(launches.values()) == (2 if in_place else 0)
        live = torch.cat([torch.arange(int(d["off"][e]), int(d["off"][e]) + int(d["n"][e])) for e in range(E)]).cuda()
        res.append([t[live], gx[live]] + g)
    assert all(torch.equal(x, y) for x, y in zip(*res))


# Weight gradients of experts with a few rows, on both tiles (every wave by itself: 128 columns by 32 rows of a 128 x 128 tile, by 64 of a 256 x 256 one).
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("E,M,Fd,rows,gap,tile", [
    (6, 136, 264, [1, 31, 32, 33, 0, 8], 0, 128),           # one and two steps of rows, tiles that end in the middle
    (4, 264, 136, [64, 63, 65, 2], 3, 128),                 # both sides of the limit in one launch
    (3, 8, 16, [5, 0, 64], 0, 128),                         # less than a lane's columns on one side
    (40, 520, 1032, [40] * 38 + [64, 0], 0, 128),           # many tiles
    (40, 512, 1024, [33 + e % 32 for e in range(39)] + [700], 0, 128),
    (64, 520, 1000, [1, 31, 32, 33, 63, 64, 65, 0] * 8, 0, 256),        # tiles that end in the middle on both sides
    (64, 1000, 520, [40, 64, 0, 65, 1, 8, 33, 90] * 8, 1, 256),
    (64, 512, 1024, [48] * 63 + [0], 0, 256),               # whole tiles
])
def test_ffn_weight_gradients_of_few_rows(E, M, Fd, rows, gap, tile, accumulate):
    """Experts of up to 64 rows, whose weight gradients are formed without the operand ring: sums of bf16 products in fp32 (64
    terms: 64 x 2^-24 of the terms' size) and one rounding to bf16, 2^-9 of the result, two where it is added to what is there."""
    from mole_amd import hip_ops as H, _lib as L
    print(f"few-row weight gradients E={E} M={M} F={Fd} rows={rows} accumulate={accumulate}", flush=True)
    d = _make(E, M, Fd, rows, torch.bfloat16, seed=E + M, pad_between=gap)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off = torch.from_numpy(d["off"]).cuda(); n = torch.from_numpy(d["n"]).cuda()
    R = max(d["R"], 1)
    assert L.lib().mole_probe_wgrad_tile(E, R, Fd, M) == tile
    h = torch.randn(R, Fd, generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    a = torch.nn.functional.gelu(h.float()).bfloat16()
    t = torch.zeros(R, Fd, dtype=torch.bfloat16, device="cuda")
    old = 0.5
    g = [torch.full_like(c[k], old) for k in ("w1", "b1", "w2", "b2")]
    H.ffn_bwd_into(c["go"], c["xd"], h, a, off, n, E, R, M, Fd, c["w1"], c["w2"], t, *g, None, accumulate, L.GELU_BWD_EXACT)
    go, xd, a64, t64 = (v.double().cpu() for v in (c["go"], c["xd"], a, t))
    for e in range(E):
        lo, hi = int(d["off"][e]), int(d["off"][e]) + int(d["n"][e])
        want = (t64[lo:hi].t() @ xd[lo:hi], t64[lo:hi].sum(0), a64[lo:hi].t() @ go[lo:hi], go[lo:hi].sum(0))
        size = (t64[lo:hi].abs().t() @ xd[lo:hi].abs(), t64[lo:hi].abs().sum(0), a64[lo:hi].abs().t() @ go[lo:hi].abs(), go[lo:hi].abs().sum(0))
        for got, w, s in zip(g, want, size):
            w = w + old if accumulate else w
            # (an expert above the limit: its larger tiles keep the same sums)
            bound = 2.0 ** -8 * w.abs() + max(hi - lo, 64) * 2.0 ** -24 * (s + old)
            assert bool(((got[e].double().cpu() - w).abs() <= bound).all())


# K-strided weights read past the caches, in a forward pass that no backward follows: from 64 MB of weights of the experts that
# can have rows, the recorded pass (256 MB) taking the ordinary loads.  Experts of a few rows on the kernel for them, of up
# to 64 and up to 128 on the tiles, of more (ordinary loads there), and of none.  The loads' cache policy changes no result.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,M,Fd,k,S", [
    (40, 1024, 1024, 1, 61), (40, 1024, 1024, 2, 120), (23, 512, 3264, 2, 33),      # few rows; the last of 67 / 134 MB
    (60, 1024, 1024, 2, 900), (60, 1024, 1024, 2, 3000), (40, 1024, 1024, 2, 4000),  # bf16 tiles: up to 64 rows, up to 128, more
    (9, 3072, 1280, 1, 301), (200, 128, 192, 1, 61), (2, 1024, 192, 1, 5), (3, 64, 192, 1, 300),      # and below the limit
])
def test_forward_only_weights_leave_no_copy(E, M, Fd, k, S, dtype):
    from mole_amd.moe.layer import MOLEModule
    print(f"forward only E={E} M={M} F={Fd} k={k} S={S} {dtype}", flush=True)
    nbytes = E * M * Fd * dtype.itemsize
    assert Fd == 192 or (64 << 20) <= nbytes < (256 << 20), "not the sizes this test is for"
    MOLEModule.reset_instances()
    m = MOLEModule(0, E, M, Fd, -1, k, 4, {"local_rank": 0, "world_size": 1, "rank": 0}, "gelu", 1, False, False, dtype=dtype)
    x = torch.randn(S, M, generator=torch.Generator().manual_seed(S)).to(dtype).cuda()
    y = m(x, capacity_factor=0.0).detach()            # recorded: the general policy
    with torch.no_grad():
        assert torch.equal(m(x, capacity_factor=0.0), y)
    f = lambda t: t.detach().float().cpu()
    r = m.last_route                                  # and against fp32 products of the experts that have rows
    want = torch.zeros(S, M)
    idx, gates, row = r.idx.cpu().long(), f(r.gates), r.row.cpu()
    assert bool((row >= 0).all())
    for e in idx.unique().tolist():
        w1, b1, w2, b2 = (f(p.all_tensors[e]) for p in (m.FC1_W_GPU, m.FC1_B_GPU, m.FC2_W_GPU, m.FC2_B_GPU))
        for j in range(k):
            t = (idx[j] == e).nonzero()[:, 0]
            a = torch.nn.functional.gelu(f(x[t.cuda()]) @ w1.t() + b1)
            want[t] += gates[j, t, None] * (a @ w2 + b2)
    assert rel_err(y, want) < tol(dtype)
    MOLEModule.reset_instances()


# bf16 widths that are multiples of 8 but not of 32: the activation by the closed forms on every kernel that takes them - 256 x
# 256 tiles (many rows and columns), 128 x 128 tiles, few rows - on every bf16 value of magnitude 2^-14 .. 8.  Error of the
# closed form 2e-6 of max(1, |h|) as in fp32 (erf and exp to a few units of fp32, amplified at most by |h|), and the result's
# rounding; -inf gives what 0 * inf gives, a NaN stays one in the derivative too.
@pytest.mark.parametrize("M,Fd,per", [(72, 29992, 1 << 20), (72, 264, 1 << 20), (200, 264, 7)])
def test_activation_at_ragged_widths_is_the_closed_form(M, Fd, per):
    from mole_amd import hip_ops as H, _lib as L
    print(f"closed-form activation M={M} F={Fd} rows per expert {per}", flush=True)
    dtype, grid = torch.bfloat16, _bf16_grid()
    rows = (grid.numel() + M - 1) // M
    vals = torch.zeros(rows * M)
    vals[:grid.numel()] = grid
    xd = vals.view(rows, M).to(dtype).cuda()
    n = [min(per, rows - lo) for lo in range(0, rows, per)]
    E = len(n)
    off = torch.tensor([0] + n).cumsum(0).int().cuda()
    n = torch.tensor(n).int().cuda()
    w1, w2 = (torch.zeros(E, Fd, M, dtype=dtype, device="cuda") for _ in range(2))
    w1[:, torch.arange(Fd), torch.arange(Fd) % M] = 1.0          # h[r, f] = xd[r, f mod M]
    w2[:, :, 0] = 1.0                                             # (go . w2^T)[r, f] = go[r, 0]
    b1, b2 = torch.zeros(E, Fd, dtype=dtype, device="cuda"), torch.zeros(E, M, dtype=dtype, device="cuda")
    go = torch.zeros(rows, M, dtype=dtype, device="cuda")
    go[:, 0] = 1.0
    out, h, a = H.ffn_fwd(xd, off, n, w1, b1, w2, b2)
    assert torch.equal(h, xd[:, torch.arange(Fd) % M])
    assert torch.equal(a[:, :M].repeat(1, Fd // M + 1)[:, :Fd], a)
    h64 = h[:, :M].double().cpu()

    def check(got, want, what):
        slack = 2e-6 * h64.abs().clamp(min=1.0)
        half_ulp = torch.pow(2.0, torch.floor(torch.log2((want.abs() + slack).clamp(min=2.0 ** -126))) - 8)
        err = (got[:, :M].double().cpu() - want).abs()
        assert bool((err <= slack + half_ulp).all()), f"{what}: {float((err / (slack + half_ulp)).max()):.1f}x its bound"

    check(a, 0.5 * h64 * (1.0 + torch.erf(h64 / 2.0 ** 0.5)), "GELU")
    g = [torch.empty_like(v) for v in (w1, b1, w2, b2)]
    t = torch.empty(rows, Fd, dtype=dtype, device="cuda")
    for fn, code in ((O.d_gelu_tanh, L.GELU_BWD_TANH), (O.d_gelu_exact, L.GELU_BWD_EXACT)):
        H.ffn_bwd_into(go, xd, h, a, off, n, E, rows, M, Fd, w1, w2, t, *g, None, False, code)
        assert torch.equal(t[:, :M].repeat(1, Fd // M + 1)[:, :Fd], t)
        check(t, fn(h64), "GELU'")
    b1[:, 0], b1[:, 1] = -float("inf"), float("nan")
    out, h, a = H.ffn_fwd(xd, off, n, w1, b1, w2, b2)
    assert bool(a[:, :2].isnan().all()) and bool(a[:, 2:].isfinite().all())
    H.ffn_bwd_into(go, xd, h, a, off, n, E, rows, M, Fd, w1, w2, t, *g, None, False, L.GELU_BWD_TANH)
    assert bool(t[:, :2].isnan().all()) and bool(t[:, 2:].isfinite().all())


def _same_class(got, want):
    """the same numbers, infinities of the same sign and NaNs in the same places (finite values are compared elsewhere)"""
    got, want = got.double().cpu(), want.double().cpu()
    code = lambda t: torch.where(t.isnan(), 3.0, torch.where(t.isposinf(), 1.0, torch.where(t.isneginf(), 2.0, 0.0)))
    return bool((code(got) == code(want)).all())


# Few-row products with an infinite weight: every row of the expert gets what fp32 arithmetic gives, an infinity of the right sign
# where the terms are one infinity and finite numbers.  Contractions of odd numbers of steps, ending inside a step, shorter
# than the waves of a block; the weight in the last piece of the contraction, in its last step and in its middle.  (Rows are
# kept from zero; the other column's term is finite.)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,M,Fd,rows", [(1, 520, 776, [9]), (4, 264, 520, [12, 12, 1, 0]), (2, 768, 2064, [3, 40]), (3, 96, 1544, [5, 24, 17])])
def test_ffn_few_rows_with_infinite_weights(E, M, Fd, rows, dtype):
    from mole_amd import hip_ops as H, _lib as L
    print(f"few rows, infinite weights E={E} M={M} F={Fd} {dtype}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=M)
    for name in ("xd", "go"):
        d[name] = torch.where(d[name].abs() < 0.1, torch.full_like(d[name], 0.1), d[name])
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    g = [torch.empty_like(d[q]).cuda() for q in ("w1", "b1", "w2", "b2")]
    owner = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    inf, R = float("inf"), d["R"]
    c = {q: (v.cuda() if torch.is_tensor(v) else v) for q, v in d.items()}
    for at in (lambda K: K - 1, lambda K: K - 9, lambda K: K // 2):
        for sign in (inf, -inf):
            w1, w2 = d["w1"].clone(), d["w2"].clone()
            w1[:, 5, at(M)], w2[:, at(Fd), 7] = sign, sign
            # h = xd.w1^T, and through the second product a finite activation on the infinite weight
            _, h, a = H.ffn_fwd(c["xd"], off, n, w1.cuda(), c["b1"], c["w2"], c["b2"])
            want = torch.einsum("rm,rfm->rf", d["xd"].double(), w1.double()[owner]) + d["b1"].double()[owner]
            assert _same_class(h, want)
            out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], w2.cuda(), c["b2"])
            want = torch.einsum("rf,rfm->rm", a.double().cpu(), w2.double()[owner]) + d["b2"].double()[owner]
            assert _same_class(out, want)
            # t = (go.w2^T) gelu'(h), gx = t.w1 with t finite
            t, gx = torch.empty(R, Fd, dtype=dtype, device="cuda"), torch.empty(R, M, dtype=dtype, device="cuda")
            H.ffn_bwd_into(c["go"], c["xd"], h, a, off, n, E, R, M, Fd, c["w1"], w2.cuda(), t, *g, None, False, L.GELU_BWD_EXACT)
            want = torch.einsum("rm,rfm->rf", d["go"].double(), w2.double()[owner]) * O.d_gelu_exact(h.double().cpu())
            assert _same_class(t, want)
            H.ffn_bwd_into(c["go"], c["xd"], h, a, off, n, E, R, M, Fd, w1.cuda(), c["w2"], t, *g, gx, False, L.GELU_BWD_EXACT)
            want = torch.einsum("rf,rfm->rm", t.double().cpu(), w1.double()[owner])
            assert _same_class(gx, want)


# out of 128 x 128 tiles that leave the CUs' second blocks idle: contractions of 84.75, 60 and 56 stages of 32, in one piece or in two planes, experts of one and of two
# m-tiles, columns that end in a tile.  bf16 results of fp32 sums in another order: the tolerance of every FFN test.
@pytest.mark.parametrize("E,M,Fd,rows", [(9, 904, 2712, [129, 256, 97, 128, 257, 200, 192, 150, 190]), (10, 640, 1920, [131, 172, 150, 129, 200] * 2), (24, 448, 1792, [140, 97, 160, 129, 90, 128] * 4)])
def test_ffn_split_contraction_of_second_blocks(E, M, Fd, rows):
    from mole_amd import hip_ops as H, _lib as L
    print(f"split contraction of second blocks E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.bfloat16, seed=E + M)
    assert L.lib().mole_ffn_workspace_bytes(L.MOLE_BF16, E, d["R"], M, Fd) == {9: 0, 10: 2, 24: 0}[E] * d["R"] * M * 4
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    out, _, a = H.ffn_fwd(c["xd"], torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda(), c["w1"], c["b1"], c["w2"], c["b2"])
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        assert rel_err(out[r], a[r].float() @ c["w2"][e].float() + c["b2"][e].float()) < tol(torch.bfloat16)


def test_ffn_split_contraction_of_more_than_2_to_18_rows():
    """The reduction of a split contraction has a block for every four rows: more of them than a grid has in y.  fp32, rows of
    eight columns; out against torch's fp32 products of the same activations (two orders of 1024 terms: 2^-24 sqrt(1024) of
    the terms' norm each)."""
    from mole_amd import hip_ops as H, _lib as L
    E, per, M, Fd = 4, 70000, 8, 1024
    R = E * per
    assert L.lib().mole_ffn_workspace_bytes(L.MOLE_F32, E, R, M, Fd) >= 2 * R * M * 4 and R / 4 > 65535
    print(f"split contraction, {R} rows", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    new = lambda *s: torch.randn(*s, device="cuda", generator=g)
    xd, w1, b1, w2, b2 = new(R, M), new(E, Fd, M), new(E, Fd), new(E, Fd, M), new(E, M)
    off = torch.arange(E + 1, dtype=torch.int32, device="cuda") * per
    n = torch.full((E,), per, dtype=torch.int32, device="cuda")
    out, _, a = H.ffn_fwd(xd, off, n, w1, b1, w2, b2)
    for e in range(E):
        ae, got = a[e * per:(e + 1) * per], out[e * per:(e + 1) * per]
        terms = (ae.norm(dim=1, keepdim=True) * w2[e].abs().max()) + b2[e].abs().max()
        assert bool(((got - (ae @ w2[e] + b2[e])).abs() <= 4 * 2.0 ** -24 * 32 * terms).all())


# fp32 tiles whose parts a block makes once: h and t (K = M: 12.5, 13 and 13.5 stages of 32 k, which the loop takes in pairs), columns that end 16
# into a tile, rows that end anywhere in one; out and gx of the last case are split into planes of 16 and 17 such stages.  Eight of k are summed
# before a rounding to nearest: 2^-24 sqrt(K / 8) in the 2-norm, as of all products by parts.  A tile that an infinite weight reaches
# is formed from fp32 operands instead, 2^-24 sqrt(K), and no other tile changes.
@pytest.mark.parametrize("E,M,Fd,rows", [(6, 400, 2064, [190, 201, 129, 128, 255, 237]), (6, 416, 2064, [190, 201, 129, 128, 255, 237]),
                                         (6, 432, 2064, [190, 201, 129, 128, 255, 237]), (8, 512, 2064, [194, 256, 130, 192, 255, 193, 129, 196])])
def test_ffn_fp32_parts_that_a_block_shares(E, M, Fd, rows):
    from mole_amd import hip_ops as H, _lib as L
    print(f"ffn fp32 shared parts E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n, R = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda(), sum(rows)
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    t, gx = torch.empty(R, Fd, device="cuda"), torch.empty(R, M, device="cuda")
    H.ffn_bwd_into(c["go"], c["xd"], h, a, off, n, E, R, M, Fd, c["w1"], c["w2"], t, *g, gx, False, L.GELU_BWD_EXACT)
    w1 = c["w1"].clone()
    w1[1, 5, M - 1] = float("inf")
    _, h_inf, _ = H.ffn_fwd(c["xd"], off, n, w1, c["b1"], c["w2"], c["b2"])
    def close(got, want, terms):
        assert float((got.double() - want).norm() / want.norm()) <= 2.0 ** -24 * terms ** 0.5
    rest = torch.arange(Fd, device="cuda") != 5
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        D = lambda q: q.double()
        want = D(c["xd"][r]) @ D(c["w1"][e]).t() + D(c["b1"][e])
        close(h[r], want, M / 8)
        close(out[r], D(a[r]) @ D(c["w2"][e]) + D(c["b2"][e]), Fd / 8)
        # (GELU' takes h to a few units of fp32 of its largest value: its share of t's error is that of as many terms)
        close(t[r], (D(c["go"][r]) @ D(c["w2"][e]).t()) * O.d_gelu_exact(D(h[r]).cpu()).cuda(), M / 8 + 16)
        close(gx[r], D(t[r]) @ D(c["w1"][e]), Fd / 8)
        if e != 1:
            assert torch.equal(h_inf[r], h[r])
        else:
            assert torch.equal(h_inf[r, 5], c["xd"][r, M - 1].sign() * float("inf"))
            close(h_inf[r][:, rest], want[:, rest], M)


# fp32 products from fp32 operands on 64-row tiles (whole and with remainders; split contractions; the last case's out on the generic
# kernel) and weight gradients, by bf16 parts of their operands: as far from 64 bits as a sum of K fp32 terms may be, 2^-24 sqrt(K) in
# the 2-norm, and with no bias: the mean error of n results is within 8 / sqrt(n) of their deviation.
@pytest.mark.parametrize("E,M,Fd,rows", [(2, 512, 1024, [1024, 1024]), (3, 272, 1040, [64, 192, 64]), (1, 1040, 132, [3200])])
def test_ffn_fp32_tiles_against_64_bits(E, M, Fd, rows):
    from mole_amd import hip_ops as H
    print(f"ffn fp32 accuracy E={E} M={M} F={Fd} rows={rows}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M + 1)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    def close(got, want, K):
        err = got.double() - want
        assert float(err.norm() / want.norm()) <= 2.0 ** -24 * K ** 0.5
        return err
    errs = []
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        errs.append(close(h[r], c["xd"][r].double() @ c["w1"][e].double().t() + c["b1"][e].double(), M).flatten())
        close(out[r], a[r].double() @ c["w2"][e].double() + c["b2"][e].double(), Fd)
        close(g[2][e], a[r].double().t() @ c["go"][r].double(), rows[e])
    err = torch.cat(errs)
    assert float(err.mean().abs()) <= 8 * float(err.std()) / err.numel() ** 0.5


# The same by parts: h and t on 128- and 64-row tiles (F = 4096, 2064), out and gx on them (M = 4096, 2064) and in planes (F = 4096: 128
# rows, 1024: 64), experts that end in half a tile and in a lone 32-row block; operands around zero and operands of one sign, whose
# terms all push the sum the same way.  Each of the
# products sums eight of k before it rounds to nearest, in units of 2^-24 of the result at most: 2^-24 sqrt(K / 8) in the 2-norm.
# What the matrix cores cut off far below the sum is 0.004 units of its last place (2^-23 at most) for every 16 of k, on a sum that
# is half of the result on average: 2^-24 times 0.004 K / 16 in the mean, for even and odd blocks of 32 rows alike.
PARTS_SHAPES = [(2, 272, 4096, [1024, 1000]), (2, 4096, 272, [1024, 1000]), (16, 144, 2064, [65] * 16), (16, 2064, 144, [65] * 16)]


@pytest.mark.parametrize("one_sign", [False, True])
@pytest.mark.parametrize("E,M,Fd,rows", PARTS_SHAPES + [(2, 2048, 1024, [288, 261])])
def test_ffn_fp32_products_drift_in_no_direction(E, M, Fd, rows, one_sign):
    from mole_amd import hip_ops as H
    print(f"ffn fp32 drift E={E} M={M} F={Fd} rows={rows} one_sign={one_sign}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    if one_sign:
        c = {k: (v.abs() if torch.is_tensor(v) else v) for k, v in c.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    flat = torch.full_like(h, 50.0)            # gelu' = 1: t = go w2^T
    gx = H.ffn_bwd(c["go"], c["xd"], flat, a, off, n, c["w1"], c["w2"], *g)

    def close(got, want, K, by_blocks=True):
        err, rms = (got.double() - want) * 2.0 ** 24, want.norm() / want.numel() ** 0.5
        assert float(err.norm() / want.norm()) <= (K / 8) ** 0.5
        odd = torch.arange(err.shape[0], device="cuda") // 32 % 2 == 1
        for e in (err[~odd], err[odd]) if by_blocks and bool(odd.any()) else (err,):
            assert float(e.mean().abs() / rms) <= 0.004 * K / 16 + 8 * float(e.std() / rms) / e.numel() ** 0.5

    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        X, A, G, W1, W2 = (t.double() for t in (c["xd"][r], a[r], c["go"][r], c["w1"][e], c["w2"][e]))
        close(h[r], X @ W1.t() + c["b1"][e].double(), M)
        close(out[r], A @ W2 + c["b2"][e].double(), Fd)
        T = G @ W2.t()
        close(gx[r], T @ W1, Fd + M)            # (t, a sum of M terms, in a sum of F)
        if rows[e] >= 128:
            close(g[2][e], A.t() @ G, rows[e])
            close(g[0][e], T.t() @ X, rows[e] + M)
            close(g[1][e][None], T.sum(0)[None], rows[e] + M, False)


# Numbers below 2^-110, where bf16 ends before the last part: the tile is computed from fp32 operands, whose error is that of K fp32
# terms.  All of an operand small; a subnormal number alone in its row, against weights that lift it.
@pytest.mark.parametrize("E,M,Fd,rows", PARTS_SHAPES)
def test_ffn_fp32_tiles_with_tiny_operands(E, M, Fd, rows):
    from mole_amd import hip_ops as H
    print(f"ffn fp32 tiny operands E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    b1, b2 = torch.zeros_like(c["b1"]), torch.zeros_like(c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    w1, w2, tiny = c["w1"] * 2.0 ** 20, c["w2"] * 2.0 ** 20, 2.0 ** -118
    _, h, a = H.ffn_fwd(c["xd"] * tiny, off, n, w1, b1, w2, b2)
    gx = H.ffn_bwd(c["go"] * tiny, c["xd"], torch.full_like(h, 50.0), a, off, n, w1, c["w2"], *g)
    sub = c["xd"].clone()
    sub[5] = 0.0
    sub[5, 7] = 2.0 ** -140
    lift = c["w1"].clone()
    lift[:, :, 7] = 2.0 ** 100
    _, hs, _ = H.ffn_fwd(sub, off, n, lift, b1, c["w2"], b2)
    assert bool((hs[5] == 2.0 ** -40).all())
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        want = (c["xd"][r] * tiny).double() @ w1[e].double().t()
        assert float((h[r].double() - want).norm() / want.norm()) <= 2.0 ** -24 * M ** 0.5
        want = (c["go"][r] * tiny).double() @ c["w2"][e].double().t() @ w1[e].double()
        assert float((gx[r].double() - want).norm() / want.norm()) <= 2.0 ** -24 * (M + Fd) ** 0.5


# Down to 2^-110 the parts hold: the last part is then a bf16 number below the smallest normal one.  Every operand of one side is between
# 2^-109 and 2^-101; the bound is that of the products by parts.
@pytest.mark.parametrize("E,M,Fd,rows", PARTS_SHAPES)
def test_ffn_fp32_parts_of_small_operands(E, M, Fd, rows):
    from mole_amd import hip_ops as H, _lib as L
    print(f"ffn fp32 small operands E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=Fd)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    small = lambda t: (t / t.abs().max() * 2.0 ** 8).abs().clamp_min(1.0).copysign(t) * 2.0 ** -109
    xd, go, b1 = small(c["xd"]), small(c["go"]), torch.zeros_like(c["b1"])
    w1, w2 = c["w1"] * 2.0 ** 20, c["w2"] * 2.0 ** 20
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    _, h, _ = H.ffn_fwd(xd, off, n, w1, b1, w2, c["b2"])
    t = torch.empty_like(h)
    H.ffn_bwd_into(go, xd, torch.full_like(h, 50.0), torch.ones_like(h), off, n, E, sum(rows), M, Fd, c["w1"], w2, t, *g, torch.empty_like(xd), False,
                   L.GELU_BWD_EXACT)
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        for got, want, K in ((h[r], xd[r].double() @ w1[e].double().t(), M), (t[r], go[r].double() @ w2[e].double().t(), M)):
            assert float((got.double() - want).norm() / want.norm()) <= 2.0 ** -24 * (K / 8) ** 0.5


# Weight gradients of experts with one row are products rounded once, those of two rows sums of two; the bias gradients are the row itself.
@pytest.mark.parametrize("E,M,Fd,rows", [(5, 132, 272, [1, 2, 1, 0, 1]), (1, 512, 140, [1])])
def test_ffn_fp32_weight_gradients_of_one_row(E, M, Fd, rows):
    from mole_amd import hip_ops as H
    print(f"ffn fp32 one row E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    a, h = torch.randn(sum(rows), Fd, device="cuda"), torch.zeros(sum(rows), Fd, device="cuda")
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        if rows[e] == 1:
            assert torch.equal(g[2][e], a[r].t() * c["go"][r]) and torch.equal(g[3][e], c["go"][r][0])
        elif rows[e] == 2:
            want = a[r].double().t() @ c["go"][r].double()
            assert float((g[2][e].double() - want).norm() / want.norm()) <= 2.0 ** -24
        else:
            assert not bool(g[2][e].any()) and not bool(g[3][e].any())


# Where a row lies in its tile makes no difference to it, and a sum of zeros is a positive zero.
@pytest.mark.parametrize("E,M,Fd,rows", PARTS_SHAPES)
def test_ffn_fp32_rows_of_a_tile_are_treated_alike(E, M, Fd, rows):
    from mole_amd import hip_ops as H
    print(f"ffn fp32 equal rows E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=Fd)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    for e in range(E):
        for t in (c["xd"], c["go"]):
            t[int(d["off"][e]):int(d["off"][e]) + rows[e]] = t[int(d["off"][e])]
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    for e in range(E):
        r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
        for t in (h, out, gx):
            assert bool((t[r] == t[int(d["off"][e])]).all())
    zero = torch.zeros_like(c["go"])
    gx = H.ffn_bwd(zero, c["xd"], torch.full_like(h, 50.0), a, off, n, c["w1"], c["w2"], *g)
    for t in (gx, *g):
        assert not bool(t.any()) and not bool(t.signbit().any())


# ... and where an operand has no finite parts the tile is computed from fp32 operands: infinities and NaNs come out as fp32
# arithmetic gives them, and a weight above the largest bf16 number gives the finite results that it should (weight gradients; the other products of
# these shapes keep fp32 operands).
@pytest.mark.parametrize("E,M,Fd,rows", [(2, 144, 272, [130, 65]), (3, 512, 528, [300, 0, 64])])
def test_ffn_fp32_tiles_with_infinite_and_largest_weights(E, M, Fd, rows):
    from mole_amd import hip_ops as H, _lib as L
    print(f"fp32 tiles, infinite weights E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M)
    for name in ("xd", "go"):
        d[name] = torch.where(d[name].abs() < 0.1, torch.full_like(d[name], 0.1), d[name])
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    owner = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    c = {q: (v.cuda() if torch.is_tensor(v) else v) for q, v in d.items()}
    g = [torch.empty_like(c[q]) for q in ("w1", "b1", "w2", "b2")]
    _, h0, a0 = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    for value in (float("inf"), -float("inf"), float("nan")):
        w1, w2, go = d["w1"].clone(), d["w2"].clone(), d["go"].clone()
        w1[:, 5, M - 1], w2[:, Fd // 2, 7], go[3, 9] = value, value, value
        _, h, _ = H.ffn_fwd(c["xd"], off, n, w1.cuda(), c["b1"], c["w2"], c["b2"])
        assert _same_class(h, torch.einsum("rm,rfm->rf", d["xd"].double(), w1.double()[owner]) + d["b1"].double()[owner])
        out, _, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], w2.cuda(), c["b2"])
        assert _same_class(out, torch.einsum("rf,rfm->rm", a.double().cpu(), w2.double()[owner]) + d["b2"].double()[owner])
        H.ffn_bwd(go.cuda(), c["xd"], h0, a0, off, n, c["w1"], c["w2"], *g)
        for e in range(E):
            r = slice(int(d["off"][e]), int(d["off"][e]) + rows[e])
            assert _same_class(g[2][e], a0[r].double().cpu().t() @ go[r].double())
    w1 = d["w1"].clone()
    w1[:, 5, 3] = 3.4e38
    x = d["xd"].clone()
    x[:, 3] = 1e-3
    _, h, _ = H.ffn_fwd(x.cuda(), off, n, w1.cuda(), c["b1"], c["w2"], c["b2"])
    want = torch.einsum("rm,rfm->rf", x.double(), w1.double()[owner]) + d["b1"].double()[owner]
    # the column of the large weight to its own scale (one term carries it), the others as any product of M terms
    assert float((h.cpu().double() - want)[:, 5].norm() / want[:, 5].norm()) <= 2.0 ** -22
    rest = torch.arange(Fd) != 5
    assert float((h.cpu().double() - want)[:, rest].norm() / want[:, rest].norm()) <= 2.0 ** -24 * M ** 0.5


@pytest.mark.parametrize("E,M,Fd,rows", PARTS_SHAPES)
def test_ffn_fp32_parts_with_infinite_and_largest_weights(E, M, Fd, rows):
    """... the products by parts, h and t (F = 4096, 2064), out and gx (M = 4096, 2064), and beside them tiles that stay with parts."""
    from mole_amd import hip_ops as H, _lib as L
    print(f"fp32 parts, infinite weights E={E} M={M} F={Fd}", flush=True)
    d = _make(E, M, Fd, rows, torch.float32, seed=M)
    R = sum(rows)
    for name in ("xd", "go", "w1", "w2"):
        d[name] = torch.where(d[name].abs() < 1e-3, torch.full_like(d[name], 1e-3), d[name])
    c = {q: (v.cuda() if torch.is_tensor(v) else v) for q, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    g = [torch.empty_like(c[q]) for q in ("w1", "b1", "w2", "b2")]
    _, h0, a0 = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    experts = [slice(int(d["off"][e]), int(d["off"][e]) + rows[e]) for e in range(E)]
    for value in (float("inf"), -float("inf"), float("nan")):
        w1, w2 = c["w1"].clone(), c["w2"].clone()
        w1[:, 5, M - 1], w2[:, Fd // 2, 7] = value, value
        _, h, _ = H.ffn_fwd(c["xd"], off, n, w1, c["b1"], c["w2"], c["b2"])
        out, _, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], w2, c["b2"])
        t, gx = torch.empty(R, Fd, device="cuda"), torch.empty(R, M, device="cuda")
        H.ffn_bwd_into(c["go"], c["xd"], h0, a0, off, n, E, R, M, Fd, c["w1"], w2, t, *g, None, False, L.GELU_BWD_EXACT)
        t_inf = t.clone()
        H.ffn_bwd_into(c["go"], c["xd"], h0, a0, off, n, E, R, M, Fd, w1, c["w2"], t, *g, gx, False, L.GELU_BWD_EXACT)
        for e, r in enumerate(experts):
            D = lambda q: q.double()
            assert _same_class(h[r], D(c["xd"][r]) @ D(w1[e]).t() + D(c["b1"][e]))
            assert _same_class(out[r], D(a[r]) @ D(w2[e]) + D(c["b2"][e]))
            assert _same_class(t_inf[r], (D(c["go"][r]) @ D(w2[e]).t()).cpu() * O.d_gelu_exact(D(h0[r]).cpu()))
            assert _same_class(gx[r], D(t[r]) @ D(w1[e]))
    # a weight above the largest bf16 number (column 5 of h to its own scale, one term carries it)
    w1 = c["w1"].clone()
    w1[:, 5, 3] = 3.4e38
    x = c["xd"].clone()
    x[:, 3] = 1e-3
    _, h, _ = H.ffn_fwd(x, off, n, w1, c["b1"], c["w2"], c["b2"])
    rest = torch.arange(Fd, device="cuda") != 5
    for e, r in enumerate(experts):
        want = x[r].double() @ w1[e].double().t() + c["b1"][e].double()
        err = h[r].double() - want
        assert float(err[:, 5].norm() / want[:, 5].norm()) <= 2.0 ** -22
        assert float(err[:, rest].norm() / want[:, rest].norm()) <= 2.0 ** -24 * M ** 0.5


# Few-row products with weights [N][K]: blocks of 32 columns and, for short contractions in many blocks, of 64 (the last two shapes; the
# 4096-column one in fp32 only, in bf16 it is the tiles'), columns that end inside either, contractions of fewer steps than a block's
# waves, of odd numbers of them and of more than a wave has in flight.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,M,Fd,rows", [(1, 24, 40, [1]), (3, 264, 72, [2, 0, 7]), (2, 520, 1048, [8, 3]), (3, 1176, 72, [2, 0, 7]),
                                         (20, 136, 4096, [1 + e % 3 for e in range(20)]), (44, 136, 1000, [1 + e % 3 for e in range(44)])])
def test_ffn_few_rows_by_block_width(E, M, Fd, rows, dtype):
    from mole_amd import hip_ops as H
    print(f"few rows, block widths E={E} M={M} F={Fd} {dtype}", flush=True)
    d = _make(E, M, Fd, rows, dtype, seed=Fd)
    c = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d.items()}
    off, n = torch.from_numpy(d["off"]).cuda(), torch.from_numpy(d["n"]).cuda()
    w_out, w_h, w_gx, *w_g = _oracle_fwd_bwd(d, "tanh")
    out, h, a = H.ffn_fwd(c["xd"], off, n, c["w1"], c["b1"], c["w2"], c["b2"])
    g = [torch.empty_like(c[k]) for k in ("w1", "b1", "w2", "b2")]
    gx = H.ffn_bwd(c["go"], c["xd"], h, a, off, n, c["w1"], c["w2"], *g)
    for got, want in zip((out, h, gx, *g), (w_out, w_h, w_gx, *w_g)):
        assert rel_err(got.float().cpu(), want) < tol(dtype)
