"""GPU parity of the DiZO projection kernels (group norms, apply, reverse)."""
import numpy as np
import pytest
import torch

from oracle import arith as A
from oracle import ref_torch as R
from oracle.arith import BF16, F16, F32, from_f32, to_f32

from tests._util import DT_TORCH, assert_bits_equal, random_theta, to_bits, to_torch

pytestmark = pytest.mark.gpu

DTS = [F16, BF16, F32]
# around the projection chunk (32768 elements) and its multiples, tiny, ragged and many-chunk groups
SIZES = [32768, 32767, 32769, 5, 64 * 64 * 5 + 3, 300000, 65536 + 8, 8191]


def _groups(dt, seed, sizes=SIZES, rel=1e-2):
    dev = torch.device("cuda", 0)
    r = np.random.default_rng(seed)
    th_h, t0_h = [], []
    for i, n in enumerate(sizes):
        t0 = random_theta(n, dt, seed + i, with_edges=False)
        th = from_f32(to_f32(t0, dt) + (r.standard_normal(n) * 0.02 * rel).astype(np.float32), dt)
        th_h.append(th)
        t0_h.append(t0)
    ths = [to_torch(x, dt, dev) for x in th_h]
    t0s = [to_torch(x, dt, dev) for x in t0_h]
    return ths, t0s, th_h, t0_h


@pytest.mark.parametrize("dt", DTS)
def test_group_norms(dt):
    from dizo_amd.table import ProjTable
    ths, t0s, th_h, t0_h = _groups(dt, 1)
    tab = ProjTable(ths, t0s)
    G = len(ths)
    dev = ths[0].device
    sumsq = torch.empty(G, dtype=torch.float64, device=dev)
    nf = torch.empty(G, dtype=torch.float32, device=dev)
    nt = torch.empty(G, dtype=DT_TORCH[dt], device=dev)
    tab.group_sumsq(sumsq, nf, nt)
    for g in range(G):
        want = A.group_sumsq(th_h[g], t0_h[g], dt)
        assert float(sumsq[g]) == pytest.approx(want, rel=1e-12)
        n_or = A.norm_from_sumsq(want, dt)
        assert abs(int(to_bits(nt[g:g + 1])[0]) - int(n_or)) <= 1
        # and within one ulp of torch.norm on the device (what the reference computes)
        tn = to_bits(torch.norm(ths[g] - t0s[g]).reshape(1))[0]
        assert abs(int(to_bits(nt[g:g + 1])[0]) - int(tn)) <= 1
    tab.close()


@pytest.mark.parametrize("dt", DTS)
def test_apply_reverse_match_oracle(dt):
    from dizo_amd._lib import DZ_PROJ_APPLY, DZ_PROJ_REVERSE, DZ_PROJ_REVERSE_SUMSQ
    from dizo_amd.table import ProjTable
    ths, t0s, th_h, t0_h = _groups(dt, 5)
    tab = ProjTable(ths, t0s)
    G = len(ths)
    dev = ths[0].device
    alphas = from_f32(np.linspace(0.85, 1.1, G).astype(np.float32), dt)
    alpha_t = to_torch(alphas, dt, dev)
    tab.project(alpha_t, DZ_PROJ_APPLY)
    app = [A.apply(th_h[g], t0_h[g], alphas[g:g + 1], dt) for g in range(G)]
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), app[g], dt, f"apply group {g}")
    sumsq = torch.empty(G, dtype=torch.float64, device=dev)
    nt = torch.empty(G, dtype=DT_TORCH[dt], device=dev)
    tab.project(alpha_t, DZ_PROJ_REVERSE_SUMSQ, sumsq=sumsq, norm_T=nt)
    rev = [A.reverse(app[g], t0_h[g], alphas[g:g + 1], dt) for g in range(G)]
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), rev[g], dt, f"reverse group {g}")
        want = A.group_sumsq(rev[g], t0_h[g], dt)
        assert float(sumsq[g]) == pytest.approx(want, rel=1e-12)
    # the fused norms equal a standalone norm pass over the same theta
    s2 = torch.empty(G, dtype=torch.float64, device=dev)
    tab.group_sumsq(s2)
    assert torch.equal(sumsq, s2)
    tab.project(alpha_t, DZ_PROJ_REVERSE)
    rev2 = [A.reverse(rev[g], t0_h[g], alphas[g:g + 1], dt) for g in range(G)]
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), rev2[g], dt, f"reverse2 group {g}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
def test_apply_reverse_match_torch_on_device(dt):
    """apply_constraints / reverse_constraints of the reference run by ROCm torch."""
    from dizo_amd._lib import DZ_PROJ_APPLY, DZ_PROJ_REVERSE
    from dizo_amd.table import ProjTable
    ths, t0s, th_h, t0_h = _groups(dt, 9, sizes=[32768, 4099, 70000])
    ref = [t.clone() for t in ths]
    G = len(ths)
    gammas = [0.9 * torch.norm(ths[g] - t0s[g]) for g in range(G)]
    alphas = R.apply_constraints(ref, t0s, gammas)
    alpha_t = torch.stack([a.reshape(()) for a in alphas]).contiguous()
    tab = ProjTable(ths, t0s)
    tab.project(alpha_t, DZ_PROJ_APPLY)
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), to_bits(ref[g]), dt, f"apply group {g}")
    R.reverse_constraints(ref, t0s, alphas)
    tab.project(alpha_t, DZ_PROJ_REVERSE)
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), to_bits(ref[g]), dt, f"reverse group {g}")
    tab.close()


def _packed_groups(dt, sizes, first):
    """Groups of odd sizes end to end in one buffer, their anchors in another from a different start
    address; (buffer, groups, anchors, their bits)."""
    ths, t0s, th_h, t0_h = _groups(dt, 77, sizes=sizes)
    total = sum(sizes)
    buf = torch.full((first + total + 9,), 3.0, dtype=DT_TORCH[dt], device="cuda")
    anchor = torch.zeros(total + 2, dtype=DT_TORCH[dt], device="cuda")
    out, out0, at = [], [], 0
    for t, t0 in zip(ths, t0s):
        buf[first + at:first + at + t.numel()] = t
        anchor[2 + at:2 + at + t.numel()] = t0
        out.append(buf[first + at:first + at + t.numel()])
        out0.append(anchor[2 + at:2 + at + t.numel()])
        at += t.numel()
    return buf, out, out0, th_h, t0_h


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("first", [1, 3])
@pytest.mark.parametrize("sizes", [[1, 7, 32768 + 5, 8193, 3, 2 * 32768, 999], [5, 1_000_001, 32768, 4096, 700_003]])
def test_packed_odd_groups_match_oracle(dt, first, sizes):
    """Norms, apply and reverse over groups that start anywhere: values against
    the oracle, sums against its fp64 sums, the elements around the groups untouched."""
    from dizo_amd._lib import DZ_PROJ_APPLY, DZ_PROJ_REVERSE_SUMSQ
    from dizo_amd.table import ProjTable
    buf, ths, t0s, th_h, t0_h = _packed_groups(dt, sizes, first)
    G = len(sizes)
    alphas = from_f32(np.linspace(0.85, 1.1, G).astype(np.float32), dt)
    alpha_t = to_torch(alphas, dt, "cuda")
    sums = [torch.empty(G, dtype=torch.float64, device="cuda") for _ in range(3)]
    tab = ProjTable(ths, t0s)
    tab.group_sumsq(sums[0])
    tab.project(alpha_t, DZ_PROJ_APPLY)
    tab.group_sumsq(sums[1])
    app = [A.apply(th_h[g], t0_h[g], alphas[g:g + 1], dt) for g in range(G)]
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), app[g], dt, f"apply group {g}")
    tab.project(alpha_t, DZ_PROJ_REVERSE_SUMSQ, sumsq=sums[2])
    rev = [A.reverse(app[g], t0_h[g], alphas[g:g + 1], dt) for g in range(G)]
    for g in range(G):
        assert_bits_equal(to_bits(ths[g]), rev[g], dt, f"reverse group {g}")
        for got, x in zip(sums, (th_h[g], app[g], rev[g])):
            # fp64 sums of n exact squares: n / 2 roundings of at most 2^-53 apart
            assert float(got[g]) == pytest.approx(A.group_sumsq(x, t0_h[g], dt), rel=max(sizes) * 2.0**-53, abs=0)
    assert bool((buf[:first] == 3.0).all()) and bool((buf[first + sum(sizes):] == 3.0).all())
    tab.close()


@pytest.mark.parametrize("dt", DTS)
def test_long_tables_match_short_ones(dt):
    """Groups that together make a long table (more than 3 * 2^24 elements), odd starts and sizes among
    them, against a table of each group by itself (a short one; the larger groups' sums take a second
    launch): the same bits from apply, fp32-alpha apply and reverse, and sums equal to the fp64 sums'
    rounding."""
    from dizo_amd import _lib as L
    from dizo_amd.table import ProjTable
    sizes = [30_000_001, 7, 12_345_678, 0, 9_000_003]
    G, total = len(sizes), sum(sizes)
    gen = torch.Generator(device="cuda").manual_seed(3)
    anchor = torch.empty(total + 1, dtype=DT_TORCH[dt], device="cuda").normal_(0, 0.02, generator=gen)
    theta = anchor + torch.empty_like(anchor).normal_(0, 4e-3, generator=gen)
    other = torch.empty_like(anchor).normal_(0, 1e-2, generator=gen)
    alpha = torch.linspace(0.85, 1.1, G, device="cuda")
    alpha_t = alpha.to(DT_TORCH[dt])
    flats, sums = [], []
    for long in (True, False):
        flat = theta.clone()
        groups, anchors = list(flat[1:].split(sizes)), list(anchor[1:].split(sizes))
        others = list(other[1:].split(sizes))
        out = torch.full((4, G), -1.0, dtype=torch.float64, device="cuda")
        for part in ([list(range(G))] if long else [[g] for g in range(G)]):
            tab = ProjTable([groups[g] for g in part], [anchors[g] for g in part])
            o, lo = out[:, part[0]:part[-1] + 1], part[0]
            hi = part[-1] + 1
            s = [torch.empty(hi - lo, dtype=torch.float64, device="cuda") for _ in range(4)]
            tab.group_dot([others[g] for g in part], s[3])
            tab.group_sumsq(s[0])
            tab.project(alpha_t[lo:hi].contiguous(), L.DZ_PROJ_APPLY)
            tab.group_sumsq(s[1])
            tab.project(alpha_t[lo:hi].contiguous(), L.DZ_PROJ_REVERSE_SUMSQ, sumsq=s[2])
            tab.project(alpha[lo:hi].contiguous(), L.DZ_PROJ_APPLY_F32ALPHA)
            for k in range(4):
                o[k] = s[k]
            tab.close()
        flats.append(flat)
        sums.append(out.cpu().numpy())
    assert torch.equal(flats[0].view(torch.int32 if dt == F32 else torch.int16), flats[1].view(torch.int32 if dt == F32 else torch.int16))
    assert float(flats[0][0]) == float(theta[0])
    np.testing.assert_allclose(sums[0][:3], sums[1][:3], rtol=max(sizes) * 2.0**-53, atol=0)
    assert (sums[0][:, 3] == 0).all() and (sums[0][:3, [0, 1, 2, 4]] > 0).all()
    # dots: against torch's fp64 sums; the terms' signs differ, so the bound is on the sum of their sizes
    for g in range(G):
        terms = others[g].double() * (theta[1:].split(sizes)[g] - anchor[1:].split(sizes)[g]).double()
        bound = float(terms.abs().sum()) * sizes[g] * 2.0**-53
        for got in (sums[0][3, g], sums[1][3, g]):
            assert abs(float(got) - float(terms.sum())) <= bound, g


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("chunks", [256, 257])
def test_sums_around_the_count_line_match_fp64(dt, chunks):
    """Short tables whose largest group has 256 chunks (counted) or 257 (a second launch adds up the chunk
    sums), 460 groups (two dot launches) with an empty one among them: norms, reverse + norms and dots
    against torch's fp64 sums. The squares are exact in fp64, so n terms are at most n / 2 roundings of
    2^-53 apart from any other order; the dots' terms differ in sign, so their bound is on their sizes."""
    from dizo_amd import _lib as L
    from dizo_amd.table import ProjTable
    cn = 2048 if dt == F32 else 4096
    sizes = [(chunks - 1) * cn + 5] + [1000 + i for i in range(457)] + [0, cn]
    G, total = len(sizes), sum(sizes)
    gen = torch.Generator(device="cuda").manual_seed(chunks)
    anchor = torch.empty(total, dtype=DT_TORCH[dt], device="cuda").normal_(0, 0.02, generator=gen)
    theta = anchor + torch.empty_like(anchor).normal_(0, 4e-3, generator=gen)
    other = torch.empty_like(anchor).normal_(0, 1e-2, generator=gen)
    ths, t0s, others = (list(x.split(sizes)) for x in (theta, anchor, other))
    tab = ProjTable(ths, t0s)
    sums, dots = (torch.full((G,), -1.0, dtype=torch.float64, device="cuda") for _ in range(2))
    alpha = torch.ones(G, dtype=DT_TORCH[dt], device="cuda")
    for mode in ("sumsq", "reverse"):
        if mode == "sumsq":
            tab.group_sumsq(sums)
        else:
            tab.project(alpha, L.DZ_PROJ_REVERSE_SUMSQ, sumsq=sums)
        tab.group_dot(others, dots)
        for g in range(G):
            d = (ths[g] - t0s[g]).double()
            assert float(sums[g]) == pytest.approx(float(d.square().sum()), rel=max(1, sizes[g]) * 2.0**-53, abs=0), (mode, g)
            terms = others[g].double() * d
            assert abs(float(dots[g]) - float(terms.sum())) <= float(terms.abs().sum()) * max(1, sizes[g]) * 2.0**-53, (mode, g)
    tab.close()


def _median_us(tab, call, passes=15):
    """Median time of the call's kernels."""
    times = []
    for _ in range(passes):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        for e in ev:
            e.record()
        tab.time_next(*ev)
        call()
        torch.cuda.synchronize()
        times.append(ev[0].elapsed_time(ev[1]) * 1e3)
    return sorted(times)[passes // 2]


@pytest.mark.parametrize("dt,elems", [(F16, 2**24), (F32, 2**23)])
def test_the_sums_of_one_large_group_do_not_hold_up_the_pass(dt, elems):
    """One group of 32 MB: the norm pass reads 64 MB, an apply moves 96. With a count for each chunk of the
    group the norms took 3.7 times the apply (58 against 15.6 us); they take about as long."""
    from dizo_amd import _lib as L
    from dizo_amd.table import ProjTable
    anchor = torch.zeros(elems, dtype=DT_TORCH[dt], device="cuda")
    tab = ProjTable([torch.full_like(anchor, 0.5)], [anchor])
    alpha, out = torch.ones(1, dtype=anchor.dtype, device="cuda"), torch.empty(1, dtype=torch.float64, device="cuda")
    apply = _median_us(tab, lambda: tab.project(alpha, L.DZ_PROJ_APPLY))
    norms = _median_us(tab, lambda: tab.group_sumsq(out))
    assert float(out[0]) == 0.25 * elems
    assert norms <= 2 * apply, (norms, apply)
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("G,lo,hi", [(66_000, 1, 200), (20_000, 2500, 2700)])
def test_many_small_groups_match_torch(dt, G, lo, hi):
    """More groups than keep counts (65,536), and groups that fill little of the long tables' chunks in a
    table of more than 3 * 2^24 elements (fp32: more than a quarter, on the persistent kernel, whose groups'
    alphas come from memory): apply and reverse against torch's own roundings, the sums against fp64 sums."""
    from dizo_amd import _lib as L
    from dizo_amd.table import ProjTable
    r = np.random.default_rng(G)
    sizes = r.integers(lo, hi + 1, size=G).tolist()
    gen = torch.Generator(device="cuda").manual_seed(G)
    t0 = torch.empty(sum(sizes), dtype=DT_TORCH[dt], device="cuda").normal_(0, 0.02, generator=gen)
    th = t0 + torch.empty_like(t0).normal_(0, 4e-3, generator=gen)
    alpha = torch.empty(G, device="cuda").uniform_(0.8, 1.2, generator=gen).to(DT_TORCH[dt])
    each = alpha.repeat_interleave(torch.tensor(sizes, device="cuda"))
    first = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    want = (th - t0) * each + t0
    tab = ProjTable(list(th.split(sizes)), list(t0.split(sizes)))
    sums = torch.empty(G, dtype=torch.float64, device="cuda")
    for mode in (L.DZ_PROJ_APPLY, L.DZ_PROJ_REVERSE_SUMSQ, L.DZ_PROJ_APPLY, L.DZ_PROJ_REVERSE):
        tab.project(alpha, mode, **({"sumsq": sums} if mode == L.DZ_PROJ_REVERSE_SUMSQ else {}))
        assert torch.equal(th.view(torch.int32 if dt == F32 else torch.int16), want.view(torch.int32 if dt == F32 else torch.int16)), mode
        if mode == L.DZ_PROJ_REVERSE_SUMSQ:
            exact = np.add.reduceat((th - t0).double().square().cpu().numpy(), first)
            np.testing.assert_allclose(sums.cpu().numpy(), exact, rtol=hi * 2.0**-53, atol=0)
        d = want - t0
        want = (d * each if mode in (L.DZ_PROJ_REVERSE, L.DZ_PROJ_REVERSE_SUMSQ) else d / each) + t0
    tab.group_sumsq(sums)
    exact = np.add.reduceat((th - t0).double().square().cpu().numpy(), first)
    np.testing.assert_allclose(sums.cpu().numpy(), exact, rtol=hi * 2.0**-53, atol=0)
    tab.close()


def test_many_small_groups_do_not_wait_one_after_another():
    """66,000 fp16 groups of 100 elements apply in at most 15 times what the same elements take in 64 groups
    (43 against 10 us; through the long tables' chunks, one small group after another, 480)."""
    from dizo_amd import _lib as L
    from dizo_amd.table import ProjTable
    total = 66_000 * 100
    th, t0 = torch.full((total,), 0.5, dtype=torch.float16, device="cuda"), torch.zeros(total, dtype=torch.float16, device="cuda")
    times = []
    for G in (66_000, 64):
        tab = ProjTable(list(th.split(total // G)), list(t0.split(total // G)))
        alpha = torch.ones(tab.n, dtype=torch.float16, device="cuda")
        times.append(_median_us(tab, lambda: tab.project(alpha, L.DZ_PROJ_APPLY)))
        tab.close()
    assert times[0] <= 15 * times[1], times


def test_empty_and_rejects():
    from dizo_amd._lib import DZ_PROJ_APPLY, DzError
    from dizo_amd.table import ProjTable
    dev = torch.device("cuda", 0)
    a = [torch.zeros(0, device=dev), torch.ones(10, device=dev)]
    b = [torch.zeros(0, device=dev), torch.zeros(10, device=dev)]
    tab = ProjTable(a, b)
    s = torch.empty(2, dtype=torch.float64, device=dev)
    tab.group_sumsq(s)
    assert s.tolist() == [0.0, 10.0]
    with pytest.raises(DzError):
        tab.project(torch.ones(3, device=dev), DZ_PROJ_APPLY)  # wrong alpha length
    with pytest.raises(DzError):
        ProjTable(a, [torch.zeros(0, device=dev), torch.zeros(11, device=dev)])
    tab.close()
    # a written tensor may not overlap another tensor or any anchor; anchors may be shared
    base = torch.zeros(40, device=dev)
    anchor = torch.zeros(10, device=dev)
    with pytest.raises(DzError, match="overlaps"):
        ProjTable([base[:10], base[5:15]], [anchor, anchor])
    with pytest.raises(DzError, match="overlaps"):
        ProjTable([base[:10], base[10:20]], [anchor, base[15:25]])
    with pytest.raises(DzError, match="overlaps"):
        ProjTable([base[:10]], [base[:10]])
    ProjTable([base[:10], base[10:20]], [anchor, anchor]).close()


@pytest.mark.parametrize("dt", DTS)
def test_apply_f32_alpha_matches_torch(dt):
    """APPLY_F32ALPHA: the reference's apply with an fp32 gamma (first-order path):
    (theta - theta0) * alpha + theta0 with alpha float32 of shape (1,), copied into T."""
    from dizo_amd._lib import DZ_PROJ_APPLY_F32ALPHA
    from dizo_amd.table import ProjTable
    ths, t0s, _, _ = _groups(dt, 13, sizes=[32768, 4099, 70000, 7, 32769])
    ref = [t.clone() for t in ths]
    G = len(ths)
    alphas = torch.tensor(np.linspace(0.5, 1.3, G), dtype=torch.float32, device=ths[0].device)
    tab = ProjTable(ths, t0s)
    tab.project(alphas, DZ_PROJ_APPLY_F32ALPHA)
    for g in range(G):
        want = ((ref[g] - t0s[g]) * alphas[g:g + 1] + t0s[g]).to(DT_TORCH[dt])
        assert_bits_equal(to_bits(ths[g]), to_bits(want), dt, f"apply_f32 group {g}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
def test_group_dot_matches_fp64(dt):
    """group_dot: sum fp32(other) * fp32(R(theta - theta0)) per group, fp64 accumulation,
    against the same sum formed in float64 by torch (up to summation order)."""
    from dizo_amd.table import ProjTable
    ths, t0s, _, _ = _groups(dt, 21, sizes=[32768, 32767, 300000, 5, 0, 8191])
    gen = torch.Generator(device="cuda").manual_seed(5)
    others = [torch.randn(t.numel(), device=t.device, generator=gen).to(DT_TORCH[dt]) for t in ths]
    G = len(ths)
    dot = torch.empty(G, dtype=torch.float64, device=ths[0].device)
    dotf = torch.empty(G, dtype=torch.float32, device=ths[0].device)
    tab = ProjTable(ths, t0s)
    tab.group_dot(others, dot, dotf)
    for g in range(G):
        delta = (ths[g] - t0s[g]).double()
        want = float((others[g].double() * delta).sum())
        assert float(dot[g]) == pytest.approx(want, rel=1e-12, abs=1e-300)
        assert float(dotf[g]) == np.float32(float(dot[g]))
    tab.close()


@pytest.mark.parametrize("large", [False, True])
def test_group_dot_more_groups_than_one_launch_takes(large):
    """500 groups (more than the 448 one dot launch takes): every group's sum
    against float64 torch, including empty groups at a batch boundary. With a
    large group in the second launch (more than 3 * 2^24 elements) the table is
    a long one, whose launches share its work counters and partial sums."""
    from dizo_amd.table import ProjTable
    dev = torch.device("cuda", 0)
    gen = torch.Generator(device=dev).manual_seed(6)
    sizes = [(1000 + 37 * i) if i not in (447, 448) else 0 for i in range(500)]
    if large:
        sizes[460] = 51_000_007
    ths = [(torch.randn(n, device=dev, generator=gen) * 0.02).half() for n in sizes]
    t0s = [(t.float() - 1e-3).half() for t in ths]
    others = [torch.randn(n, device=dev, generator=gen).half() for n in sizes]
    dot = torch.empty(500, dtype=torch.float64, device=dev)
    tab = ProjTable(ths, t0s)
    tab.group_dot(others, dot)
    for g in range(500):
        terms = others[g].double() * (ths[g] - t0s[g]).double()
        want = float(terms.sum())
        # the large group's 5e7 terms all but cancel (sum 7, sizes 4e4): bounded by their sizes
        near = 0.0 if sizes[g] < 10**6 else float(terms.abs().sum()) * sizes[g] * 2.0**-53
        assert float(dot[g]) == pytest.approx(want, rel=1e-12, abs=max(near, 1e-300)), g
    tab.close()


@pytest.mark.parametrize("dt", [F16, F32])
def test_more_groups_than_the_lds_alpha_table(dt):
    """More groups (4100, and a large one that makes the table a long one) than
    a workgroup of the persistent projection kernel keeps alphas for in LDS
    (4096): each chunk then reads its group's alpha from memory. Apply, reverse
    and the group norms against the oracle, on views of one buffer (the large
    group against torch's roundings)."""
    from dizo_amd._lib import DZ_PROJ_APPLY, DZ_PROJ_REVERSE, DZ_PROJ_REVERSE_SUMSQ
    from dizo_amd.table import ProjTable
    G, n = 4100, 37
    dev = torch.device("cuda", 0)
    r = np.random.default_rng(3)
    t0_all = random_theta(G * n, dt, 7, with_edges=False)
    th_all = from_f32(to_f32(t0_all, dt) + (r.standard_normal(G * n) * 2e-4).astype(np.float32), dt)
    th_buf, t0_buf = to_torch(th_all, dt, dev), to_torch(t0_all, dt, dev)
    ths = [th_buf[g * n:(g + 1) * n] for g in range(G)]
    t0s = [t0_buf[g * n:(g + 1) * n] for g in range(G)]
    alphas = from_f32(np.linspace(0.6, 1.2, G + 1).astype(np.float32), dt)
    alpha_t = to_torch(alphas, dt, dev)
    gen = torch.Generator(device="cuda").manual_seed(4)
    t0_large = torch.empty(3 * 2**24 + 10_000_019, dtype=DT_TORCH[dt], device=dev).normal_(0, 0.02, generator=gen)
    large = t0_large + torch.empty_like(t0_large).normal_(0, 4e-3, generator=gen)
    want_large = (large - t0_large) * alpha_t[G:] + t0_large
    tab = ProjTable(ths + [large], t0s + [t0_large])
    tab.project(alpha_t, DZ_PROJ_APPLY)
    assert torch.equal(large, want_large)
    got = to_bits(th_buf)
    want = np.concatenate([A.apply(th_all[g * n:(g + 1) * n], t0_all[g * n:(g + 1) * n], alphas[g:g + 1], dt)
                           for g in range(G)])
    assert_bits_equal(got, want, dt, "apply")
    sumsq = torch.empty(G + 1, dtype=torch.float64, device=dev)
    tab.project(alpha_t, DZ_PROJ_REVERSE_SUMSQ, sumsq=sumsq)
    want_large = (want_large - t0_large) / alpha_t[G:] + t0_large
    assert torch.equal(large, want_large)
    exact = float((large - t0_large).double().square().sum())
    assert float(sumsq[G]) == pytest.approx(exact, rel=large.numel() * 2.0**-53)
    rev = [A.reverse(want[g * n:(g + 1) * n], t0_all[g * n:(g + 1) * n], alphas[g:g + 1], dt) for g in range(G)]
    assert_bits_equal(to_bits(th_buf), np.concatenate(rev), dt, "reverse")
    s = sumsq.cpu().numpy()
    for g in range(0, G, 97):
        assert s[g] == pytest.approx(A.group_sumsq(rev[g], t0_all[g * n:(g + 1) * n], dt), rel=1e-12), g
    tab.project(alpha_t, DZ_PROJ_REVERSE)
    rev = [A.reverse(rev[g], t0_all[g * n:(g + 1) * n], alphas[g:g + 1], dt) for g in range(G)]
    assert_bits_equal(to_bits(th_buf), np.concatenate(rev), dt, "reverse without norms")
    assert torch.equal(large, (want_large - t0_large) / alpha_t[G:] + t0_large)
    tab.close()


def _edge_alphas(dt):
    """Alphas across the range: subnormal ones (for bf16, 1 / alpha overflows
    below 2^-128), the smallest normal, tiny, typical, huge and negative
    values, and random ratios near 1."""
    r = np.random.default_rng(17)
    vals = [2.0 ** -126, 2.0 ** -100, 2.0 ** -64, 1e-8, 1e-3, 0.5, 0.9, 1.0, 1.1, 2.0, 3.0, 7.0, 1e3, 2.0 ** 60,
            -0.75, -3.0] + list(r.uniform(0.5, 2.0, 16))
    bits = [int(b) for b in from_f32(np.array(vals, dtype=np.float32), dt)]
    if dt == BF16:
        bits += [0x0001, 0x0040, 0x007f, 0x0080, 0x7f7f]  # subnormals, min normal, max
    else:
        bits += [0x0001, 0x0200, 0x03ff, 0x0400, 0x7bff]
    out = []
    for b in bits:
        v = float(to_f32(np.array([b], dtype=A.BITS_DTYPE[dt]), dt)[0])
        if v != 0 and np.isfinite(v) and b not in out:
            out.append(b)
    return np.array(out, dtype=A.BITS_DTYPE[dt])


@pytest.mark.parametrize("dt", [BF16, F16])
def test_reverse_every_dividend_matches_oracle(dt):
    """reverse and reverse+norm with theta0 = 0 and theta running through all
    65536 16-bit patterns (inf, NaN, subnormals and zeros included), so the
    quotient R_T(R_T(theta - theta0) / alpha) meets every dividend, for ~40
    alphas from subnormal to huge: bit for bit against the oracle's IEEE
    division (the bf16 kernel divides by multiplying with fp32(1 / alpha),
    falling back to the division where that could round differently)."""
    from dizo_amd._lib import DZ_PROJ_REVERSE, DZ_PROJ_REVERSE_SUMSQ
    from dizo_amd.table import ProjTable
    dev = torch.device("cuda", 0)
    alphas = _edge_alphas(dt)
    G = len(alphas)
    every = np.arange(65536, dtype=np.uint32).astype(A.BITS_DTYPE[dt])
    zeros = np.zeros(65536, dtype=A.BITS_DTYPE[dt])
    ths = [to_torch(every, dt, dev) for _ in range(G)]
    t0s = [to_torch(zeros, dt, dev) for _ in range(G)]
    tab = ProjTable(ths, t0s)
    alpha_t = to_torch(alphas, dt, dev)
    for mode, what in ((DZ_PROJ_REVERSE, "reverse"), (DZ_PROJ_REVERSE_SUMSQ, "reverse+norm")):
        for t in ths:
            t.copy_(to_torch(every, dt, dev))
        if mode == DZ_PROJ_REVERSE_SUMSQ:
            sumsq = torch.empty(G, dtype=torch.float64, device=dev)
            tab.project(alpha_t, mode, sumsq=sumsq)
        else:
            tab.project(alpha_t, mode)
        for g in range(G):
            want = A.reverse(every, zeros, alphas[g:g + 1], dt)
            assert_bits_equal(to_bits(ths[g]), want, dt, f"{what}, alpha bits {hex(int(alphas[g]))}")
    tab.close()
