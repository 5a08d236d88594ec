"""GPU parity of the ZO step kernels (perturb / update / restore+update / z export).

Compared bit for bit against
  * the numpy oracle (oracle.arith + oracle.rng computes z itself), and
  * torch on the ROCm device evaluating the reference's expressions
    (oracle.ref_torch) fed the z exported by the library.
"""
import numpy as np
import pytest
import torch

from oracle import arith as A
from oracle import ref_torch as R
from oracle import rng
from oracle.arith import BF16, F16, F32

from tests._util import DT_TORCH, assert_bits_equal, random_theta, to_bits, to_torch

pytestmark = pytest.mark.gpu

DTS = [F16, BF16, F32]
# sizes: tiny, odd, group-aligned, one chunk (32768), chunk + 1, several chunks
SIZES = [1, 7, 8, 9, 1000, 32768, 32769, 3 * 50000, 65536 + 24, 2050 * 64, 0, 5]


def _make_tensors(dt, seed, sizes=SIZES, misaligned=(3, 6)):
    """Device tensors with oracle-generated contents; some are views whose data
    pointer is not 16-byte aligned."""
    dev = torch.device("cuda", 0)
    tensors, host = [], []
    keep = []
    for i, n in enumerate(sizes):
        bits = random_theta(n, dt, seed + i) if n else np.zeros(0, A.BITS_DTYPE[dt])
        t = to_torch(bits, dt, dev)
        if i in misaligned and n:
            buf = torch.empty(n + 1, dtype=t.dtype, device=dev)
            view = buf[1:]
            view.copy_(t)
            keep.append(buf)
            t = view
        tensors.append(t)
        host.append(bits)
    return tensors, host, keep


def _fused_table(tensors, prefetch, **kw):
    """A ZO table on the long tables' kernel, whose restore+update+next perturb
    launches run the prefetching tile loop (prefetch=True, every launch) or the
    plain tile loop (prefetch=False, no launch); prefetch=None: on the kernel
    that its size gives it, the short tables' one for most sizes here."""
    from dizo_amd.table import ZOTable
    tab = ZOTable(tensors, **kw)
    if prefetch is not None:
        tab.set_prefetch_min_tiles(1 if prefetch else 0xFFFFFFFF)
    return tab


def _z_host(table, seed, dt):
    return [rng.tensor_z_bits(seed, off, n, dt) for off, n in zip(table.z_offsets, table.numels)]


@pytest.mark.parametrize("dt", DTS)
def test_z_export_matches_oracle(dt):
    from dizo_amd.table import ZOTable, normals
    tensors, _, keep = _make_tensors(dt, 100)
    tab = ZOTable(tensors)
    seed = 987654321
    for i, t in enumerate(tensors):
        z = tab.export_z(seed, i)
        assert_bits_equal(to_bits(z).ravel(), rng.tensor_z_bits(seed, tab.z_offsets[i], t.numel(), dt), dt,
                          f"export z tensor {i}")
    # dense normals at an unaligned offset and in the gamma stream
    for stream, off in ((0, 13), (1, 0), (2, 2**33 + 5)):
        z = normals(seed, stream, off, 5000, DT_TORCH[dt], torch.device("cuda", 0))
        assert_bits_equal(to_bits(z), rng.z_bits(seed, stream, np.arange(5000, dtype=np.uint64) + np.uint64(off), dt),
                          dt, f"normals stream {stream}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("offset,n", [(5, 3), (7, 2), (0, 8), (3, 2**19 - 11), (0, 2**19 - 8), (1, 2**19 - 1), (8, 2**19),
                                      (2**35 - 8 * 700 + 3, 2**19 + 13), (0, 2**22 + 5), (2**64 - 8 * 9 + 2, 4096)])
def test_normals_ranges_match_oracle(dt, offset, n):
    """Ranges that start and end inside a Philox block, on both sides of 2^16 blocks (where the LDS
    kernel takes over), across a wrap of the counter's low word and of the element index."""
    from dizo_amd.table import normals
    z = normals(99, 0, offset, n, DT_TORCH[dt], torch.device("cuda", 0))
    idx = np.arange(n, dtype=np.uint64) + np.uint64(offset)
    assert_bits_equal(to_bits(z), rng.z_bits(99, 0, idx, dt), dt, f"normals {offset} {n}")


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("n", [100, 2**19 + 3])
def test_normals_into_a_misaligned_buffer(dt, n):
    """z written one element past a vector boundary leaves its neighbours alone."""
    from dizo_amd import _lib as L
    from dizo_amd.table import dtype_code
    buf = torch.full((n + 2,), 7.0, dtype=DT_TORCH[dt], device="cuda")
    L.call("dz_normals", 5, 1, 11, n, dtype_code(buf.dtype), buf[1:].data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert float(buf[0]) == 7.0 and float(buf[-1]) == 7.0
    assert_bits_equal(to_bits(buf[1:-1]), rng.z_bits(5, 1, np.arange(n, dtype=np.uint64) + np.uint64(11), dt), dt)


def test_philox_blocks_match_oracle():
    from dizo_amd.table import philox_blocks
    for seed, stream, q0 in ((0, 0, 0), (26, 1, 2**32 - 3), (2**64 - 1, 2, 2**40)):
        got = philox_blocks(seed, stream, q0, 4096, torch.device("cuda", 0)).cpu().numpy().view(np.uint32)
        want = rng.philox_groups(seed, stream, np.arange(4096, dtype=np.uint64) + np.uint64(q0))
        np.testing.assert_array_equal(got, want)


def test_normals_and_philox_take_the_device_in_every_form():
    from dizo_amd.table import normals, philox_blocks
    z, w = normals(3, 1, 5, 100, torch.float16, torch.device("cuda", 0)), philox_blocks(3, 1, 5, 9, torch.device("cuda", 0))
    for device in (0, "cuda", "cuda:0", torch.device("cuda")):
        assert torch.equal(normals(3, 1, 5, 100, torch.float16, device), z)
        assert torch.equal(philox_blocks(3, 1, 5, 9, device), w)
    with torch.device("cuda"):  # the default device
        assert torch.equal(normals(3, 1, 5, 100, torch.float16, None), z)
        assert torch.equal(philox_blocks(3, 1, 5, 9, None), w)


@pytest.mark.parametrize("dt", DTS)
def test_rmw_uses_exported_z(dt):
    """theta = 0, scale 1, eps 1 leaves exactly z: the kernel's in-register z is the exported z."""
    from dizo_amd.table import ZOTable
    dev = torch.device("cuda", 0)
    tensors = [torch.zeros(n, dtype=DT_TORCH[dt], device=dev) for n in (5, 40000, 32768 * 3 + 7)]
    tab = ZOTable(tensors)
    tab.perturb(31337, 1.0, 1.0)
    for i, t in enumerate(tensors):
        assert_bits_equal(to_bits(t), to_bits(tab.export_z(31337, i)).ravel(), dt, f"tensor {i}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("prefetch", [True, False, None])
@pytest.mark.parametrize("first", [1, 3, 7])
def test_packed_odd_tensors_match_oracle(dt, prefetch, first):
    """Tensors of odd sizes end to end in one buffer, from every kind of start address, full tiles
    among them: every pass against the oracle, and the elements around the tensors untouched."""
    sizes = [1, 7, 24576 + 5, 8193, 2 * 32768 + 1, 3, 32768, 999]
    buf = torch.full((first + sum(sizes) + 9,), 3.0, dtype=DT_TORCH[dt], device="cuda")
    tensors, host, at = [], [], first
    for i, n in enumerate(sizes):
        bits = random_theta(n, dt, 900 + i)
        buf[at:at + n] = to_torch(bits, dt, "cuda")
        tensors.append(buf[at:at + n])
        host.append(bits)
        at += n
    tab = _fused_table(tensors, prefetch)
    s1, s2, eps, g, lr = 5, 6, 1e-3, 0.75, 1e-3
    tab.perturb(s1, -2.0, eps)
    tab.restore_update_perturb(s1, s2, eps, g, lr)
    tab.restore_update(s2, eps, g, lr)
    tab.update(s1, g, lr)
    for i, (t, h, z1, z2) in enumerate(zip(tensors, host, _z_host(tab, s1, dt), _z_host(tab, s2, dt))):
        h = A.perturb(A.restore_update(A.perturb(h, z1, -2, eps, dt), z1, eps, g, lr, dt), z2, 1, eps, dt)
        h = A.update(A.restore_update(h, z2, eps, g, lr, dt), z1, g, lr, dt)
        assert_bits_equal(to_bits(t), h, dt, f"tensor {i}")
    assert bool((buf[:first] == 3.0).all()) and bool((buf[at:] == 3.0).all())
    tab.close()


# the lines up to which the three-way pass, restore + update, and perturb and update run the short tables' kernel
SHORT_LINES = {F16: (5 * 2**22, 3 * 2**24, 2**26), BF16: (3 * 2**22, 3 * 2**23, 2**26), F32: (2**24,)}


@pytest.mark.parametrize("dt,elems", [(dt, n) for dt in DTS for n in (8192 * 256 - 3, 8192 * 1500 + 77, *SHORT_LINES[dt])])
def test_short_tables_match_the_persistent_kernel(dt, elems):
    """Tables below and on the lines up to which passes run the short tables' kernel (at least one pass does
    at each size), with one to many tiles per workgroup and odd tensors among them, across a wrap of the z
    counter's low word: every pass gives the persistent kernel's bits (which the other tests hold against
    the oracle)."""
    from dizo_amd.table import ZOTable
    cut = [elems // 3 + 1, 5, elems // 2 + 3]
    sizes = cut + [elems - sum(cut)]
    gen = torch.Generator(device="cuda").manual_seed(elems)
    start = (torch.randn(elems, device="cuda", generator=gen) * 0.02).to(DT_TORCH[dt])
    offs, z = [], 2**35 - 8 * (elems // 16)
    for n in sizes:
        offs.append(z)
        z += (n + 7) // 8 * 8
    out = []
    for short in (True, False):
        flat = start.clone()
        tab = ZOTable(list(flat.split(sizes)), z_offsets=offs) if short else _fused_table(list(flat.split(sizes)), True, z_offsets=offs)
        tab.perturb(1, -2.0, 1e-3)
        tab.restore_update_perturb(1, 2, 1e-3, 0.3, 1e-2)
        tab.restore_update(2, 1e-3, -0.7, 1e-2)
        tab.update(3, 1.25, 1e-2)
        out.append(to_bits(flat))
        tab.close()
    assert_bits_equal(out[0], out[1], dt, f"{elems} elements")


def _median_us(tab, call, passes=25):
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


def test_prefetch_min_tiles_of_0_restores_the_short_kernel():
    """2^20 fp16 elements: a pass of the short tables' kernel takes 4 us, of the long tables' one 10 to 14.
    The default may be set again, also after another value."""
    from dizo_amd.table import ZOTable
    tab = ZOTable([torch.zeros(2**20, dtype=torch.float16, device="cuda")])

    def time():
        return _median_us(tab, lambda: tab.restore_update_perturb(1, 2, 1e-3, 0.3, 1e-3))

    time()
    default = time()
    for tiles, same in ((0, True), (1, False), (0, True)):
        tab.set_prefetch_min_tiles(tiles)
        assert (time() < 1.4 * default) == same, tiles
    tab.close()


def test_tensors_a_little_over_a_tile_share_out_evenly():
    """1,200 tensors of a full short tile (8,192 elements) and 8 elements more: the short tables' kernel is
    no slower than the long tables' one (17.0 against 19.6 us; with the full tiles all on one half of the
    workgroups it took 25.1)."""
    from dizo_amd.table import ZOTable
    tab = ZOTable(list(torch.zeros(1200 * 8200, dtype=torch.bfloat16, device="cuda").split(8200)))
    times = []
    for long_kernel in (False, True):
        if long_kernel:
            tab.set_prefetch_min_tiles(1)
        call = lambda: tab.restore_update_perturb(1, 2, 1e-3, 0.3, 1e-3)  # noqa: E731
        _median_us(tab, call, 3)
        times.append(_median_us(tab, call))
    assert times[0] <= 1.1 * times[1], times
    tab.close()


@pytest.mark.parametrize("dt", DTS)
def test_tables_around_the_cache_size_agree(dt):
    """The same elements in a table of 256 MB (plain accesses), in one a little longer (streaming
    accesses) and in slices below the short-table line: the same bits from every pass."""
    from dizo_amd.table import ZOTable
    n = 2**28 // DT_TORCH[dt].itemsize
    gen = torch.Generator(device="cuda").manual_seed(11)
    start = torch.empty(n + 12345, dtype=DT_TORCH[dt], device="cuda").normal_(0.0, 0.02, generator=gen)

    def run(lo, hi):
        flat = start[lo:hi].clone()
        tab = ZOTable([flat], z_offsets=[lo])
        tab.perturb(1, -2.0, 1e-3)
        tab.restore_update_perturb(1, 2, 1e-3, 0.3, 1e-2)
        tab.restore_update(2, 1e-3, -0.7, 1e-2)
        tab.update(3, 1.25, 1e-2)
        tab.close()
        return flat.view(torch.int32 if dt == F32 else torch.int16)

    plain, streamed = run(0, n), run(0, n + 12345)
    assert torch.equal(plain, streamed[:n])
    for lo in (0, n // 2 + 8, n - 2**20):
        assert torch.equal(plain[lo:lo + 2**20], run(lo, lo + 2**20)), lo


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("scale", [1.0, -2.0, 0.5])
@pytest.mark.parametrize("prefetch", [True, None])
def test_perturb_matches_oracle(dt, scale, prefetch):
    tensors, host, keep = _make_tensors(dt, 7)
    tab = _fused_table(tensors, prefetch)
    seed, eps = 123456789, 1e-3
    tab.perturb(seed, scale, eps)
    for i, (t, h, z) in enumerate(zip(tensors, host, _z_host(tab, seed, dt))):
        assert_bits_equal(to_bits(t).ravel(), A.perturb(h, z, scale, eps, dt), dt, f"tensor {i} n={h.size}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("prefetch", [True, None])
def test_full_step_sequence_matches_oracle(dt, prefetch):
    """perturb +1, -2, then fused restore+update; and the unfused restore, update."""
    tensors, host, keep = _make_tensors(dt, 21)
    tab = _fused_table(tensors, prefetch)
    seed, eps, g, lr = 424242, 1e-3, -0.734375, 9.93875e-07
    zs = _z_host(tab, seed, dt)
    tab.perturb(seed, 1.0, eps)
    tab.perturb(seed, -2.0, eps)
    want = [A.perturb(A.perturb(h, z, 1, eps, dt), z, -2, eps, dt) for h, z in zip(host, zs)]
    for i, (t, w) in enumerate(zip(tensors, want)):
        assert_bits_equal(to_bits(t).ravel(), w, dt, f"after -2, tensor {i}")
    clones = [t.clone() for t in tensors]
    tab.restore_update(seed, eps, g, lr)
    final = [A.restore_update(w, z, eps, g, lr, dt) for w, z in zip(want, zs)]
    for i, (t, w) in enumerate(zip(tensors, final)):
        assert_bits_equal(to_bits(t).ravel(), w, dt, f"fused, tensor {i}")
    # the unfused path on the clones gives the same bits
    for t, c in zip(tensors, clones):
        t.copy_(c)
    tab.perturb(seed, 1.0, eps)
    tab.update(seed, g, lr)
    for i, (t, w) in enumerate(zip(tensors, final)):
        assert_bits_equal(to_bits(t).ravel(), w, dt, f"unfused, tensor {i}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("prefetch", [False, True, None])
def test_restore_update_perturb_matches_oracle(dt, prefetch):
    """Restore + update of step seed, then +1 of step next_seed, in one pass: the
    same bits as the three passes, and as the oracle (plain and prefetching
    tile loops)."""
    from dizo_amd.table import ZOTable
    tensors, host, keep = _make_tensors(dt, 61)
    clones = [t.clone() for t in tensors]
    tab = _fused_table(tensors, prefetch)
    seed, nxt, eps, g, lr = 9090, 9091, 1e-3, 0.6875, 9.9e-07
    tab.restore_update_perturb(seed, nxt, eps, g, lr)
    z1, z2 = _z_host(tab, seed, dt), _z_host(tab, nxt, dt)
    for i, (t, h) in enumerate(zip(tensors, host)):
        want = A.perturb(A.restore_update(h, z1[i], eps, g, lr, dt), z2[i], 1, eps, dt)
        assert_bits_equal(to_bits(t).ravel(), want, dt, f"fused3 tensor {i}")
    tab2 = ZOTable(clones)
    tab2.restore_update(seed, eps, g, lr)
    tab2.perturb(nxt, 1.0, eps)
    for i, (t, c) in enumerate(zip(tensors, clones)):
        assert_bits_equal(to_bits(t).ravel(), to_bits(c).ravel(), dt, f"fused3 vs two passes, tensor {i}")
    tab.close()
    tab2.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("prefetch", [True, None])
def test_device_scalar_overrides(dt, prefetch):
    """Seed / grad / lr read from device memory give the by-value results."""
    tensors, host, keep = _make_tensors(dt, 33, sizes=[40000, 77])
    tab = _fused_table(tensors, prefetch)
    seed, eps, g, lr = 55555, 1e-3, 1.25, 2e-6
    dev = torch.device("cuda", 0)
    d_seed = torch.tensor([seed], dtype=torch.int64, device=dev)
    d_grad = torch.tensor(g, dtype=DT_TORCH[dt], device=dev)
    d_lr = torch.tensor(lr, dtype=torch.float32, device=dev)
    tab.perturb(0, 1.0, eps, d_seed=d_seed)
    tab.restore_update(1, eps, 0.0, 0.0, d_seed=d_seed, d_grad=d_grad, d_lr=d_lr)
    zs = _z_host(tab, seed, dt)
    for i, (t, h, z) in enumerate(zip(tensors, host, zs)):
        want = A.restore_update(A.perturb(h, z, 1, eps, dt), z, eps, g, lr, dt)
        assert_bits_equal(to_bits(t).ravel(), want, dt, f"tensor {i}")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
def test_matches_torch_on_device(dt):
    """The reference's own expressions evaluated by ROCm torch, fed the exported z."""
    from dizo_amd.table import ZOTable
    tensors, host, keep = _make_tensors(dt, 40, sizes=[1, 9, 32769, 100000], misaligned=())
    ref = [t.clone() for t in tensors]
    tab = ZOTable(tensors)
    seed, eps, g, lr = 777, 1e-3, 3.5, 1e-6
    zs = [tab.export_z(seed, i) for i in range(len(tensors))]
    for s in (1, -2, 1):
        tab.perturb(seed, float(s), eps)
        R.zo_perturb_parameters(ref, zs, s, eps)
        for i, (t, r) in enumerate(zip(tensors, ref)):
            assert_bits_equal(to_bits(t), to_bits(r), dt, f"s={s} tensor {i}")
    tab.update(seed, g, lr)
    R.zo_update(ref, zs, g, lr)
    for i, (t, r) in enumerate(zip(tensors, ref)):
        assert_bits_equal(to_bits(t), to_bits(r), dt, f"update tensor {i}")
    tab.close()


def _opt_like_sizes(target_elems: int, d: int = 768):
    """Tensor sizes in OPT layer order (matrices, biases, layer norms) up to target_elems."""
    out, total = [2050 * d], 2050 * d
    while total < target_elems:
        layer = [d * d, d] * 4 + [d, d, 4 * d * d, 4 * d, 4 * d * d, d, d, d]
        out += layer
        total += sum(layer)
    return out + [d, d]


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("target", [200_000, 1_200_000, 6_000_000, 90_000_000])
@pytest.mark.parametrize("prefetch", [False, True, None])
def test_multi_tile_launches_match_torch(dt, target, prefetch):
    """Tables of 3 to ~1400 tiles (grids below and above the counter fan-out,
    several tiles per workgroup): every element is processed exactly once per
    launch, also on consecutive launches (the work counters reset themselves).
    Checked against the reference's expressions run by ROCm torch with the
    exported z; the fused three-way pass on the plain and the prefetching
    tile loop."""
    dev = torch.device("cuda", 0)
    sizes = _opt_like_sizes(target, d=64 if target < 1_000_000 else 768)
    print(f"dt={dt} target={target} prefetch={prefetch} tensors={len(sizes)} elems={sum(sizes)}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(target)
    tensors = [(torch.randn(n, device=dev, generator=gen) * 0.02).to(DT_TORCH[dt]) for n in sizes]
    ref = [t.clone() for t in tensors]
    tab = _fused_table(tensors, prefetch)
    seed, eps, g, lr = 1000 + target % 977, 1e-3, -2.25, 1e-6
    zs = [tab.export_z(seed, i) for i in range(len(tensors))]
    for s_ in (1, -2):
        tab.perturb(seed, float(s_), eps)
        R.zo_perturb_parameters(ref, zs, s_, eps)
    tab.restore_update(seed, eps, g, lr)
    R.zo_perturb_parameters(ref, zs, 1, eps)
    R.zo_update(ref, zs, g, lr)
    tab.update(seed, g, lr)
    R.zo_update(ref, zs, g, lr)
    seed2 = seed + 1
    zs2 = [tab.export_z(seed2, i) for i in range(len(tensors))]
    tab.restore_update_perturb(seed, seed2, eps, g, lr)
    R.zo_perturb_parameters(ref, zs, 1, eps)
    R.zo_update(ref, zs, g, lr)
    R.zo_perturb_parameters(ref, zs2, 1, eps)
    torch.cuda.synchronize()
    bad = [i for i, (t, r) in enumerate(zip(tensors, ref)) if not torch.equal(t.view(torch.int16 if dt != F32 else torch.int32),
                                                                           r.view(torch.int16 if dt != F32 else torch.int32))]
    assert not bad, f"{len(bad)} tensors differ, first {bad[:5]}"
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("divisor", [2 * 1e-3, 2 * 0.1, 0.003, 0.7, 3.0])
def test_projected_grad_device_rule(dt, divisor):
    """torch on the device divides a T tensor by a python scalar as the oracle's
    device rule says: R_T(x * fp32(1 / divisor)) with the reciprocal taken in double."""
    r = np.random.default_rng(2)
    l1 = A.from_f32((r.random(4096) * 3).astype(np.float32), dt)
    l2 = A.from_f32((r.random(4096) * 3).astype(np.float32), dt)
    dev = torch.device("cuda", 0)
    got = to_bits((to_torch(l1, dt, dev) - to_torch(l2, dt, dev)) / divisor)
    d = A.from_f32(A.to_f32(l1, dt) - A.to_f32(l2, dt), dt)
    assert_bits_equal(got, A.scalar_div_device(d, divisor, dt), dt, f"device scalar div by {divisor}")


def test_stale_table_raises():
    from dizo_amd._lib import DzError
    from dizo_amd.table import ZOTable
    p = torch.nn.Parameter(torch.zeros(100, device="cuda"))
    tab = ZOTable([p.data])
    p.data = torch.ones(100, device="cuda")  # rebinding, as trainer.py:1442 does
    tab.tensors[0] = p.data
    with pytest.raises(DzError):
        tab.check()
    tab.close()


def test_rejects_bad_inputs():
    from dizo_amd._lib import DzError
    from dizo_amd.table import ZOTable
    with pytest.raises(DzError):
        ZOTable([torch.zeros(4)])  # CPU tensor
    with pytest.raises(DzError):
        ZOTable([torch.zeros(4, device="cuda"), torch.zeros(4, device="cuda", dtype=torch.float16)])
    with pytest.raises(DzError):
        ZOTable([torch.zeros(4, 4, device="cuda").t()])  # non-contiguous
    # overlapping tensors would be read and written by two workgroups at once
    base = torch.zeros(100, device="cuda")
    with pytest.raises(DzError, match="overlaps"):
        ZOTable([base[:60], base[50:]])
    with pytest.raises(DzError, match="overlaps"):
        ZOTable([base, base[10:20]])
    with pytest.raises(DzError, match="overlaps"):
        ZOTable([base, base])
    ZOTable([base[:50], base[50:]]).close()  # adjacent is fine


def _fp16_tie_values(lr: float) -> np.ndarray:
    """Positive fp16 values c below 64 whose fp32 product with fp32(lr) lies
    exactly halfway between two fp16 values: rounding that fp32 product to
    fp16 (torch's opmath recipe) and rounding the exact product once give
    different results."""
    cand = np.arange(1, 0x5400, dtype=np.uint16).view(np.float16)
    lr32 = np.float32(lr)
    twice = (cand.astype(np.float32) * lr32).astype(np.float16)
    once = (cand.astype(np.float64) * np.float64(lr32)).astype(np.float16)
    return cand[twice.view(np.int16) != once.view(np.int16)]


def test_update_rounds_ties_like_torch_cpu_and_cuda():
    """lr * c for fp16 c whose fp32 product is exactly halfway between two fp16
    values (lr = 9.15e-07, the learning rate where a C3-shape run against ROCm
    torch first separated, at a 2,560-element bias).

    * The library's update rounds the fp32 product to even, as torch on the
      CPU does (and CUDA, whose opmath kernels compute in fp32 and round the
      result): bit for bit against torch on the CPU.
    * ROCm torch's own fp16 `scalar * tensor` kernel is run on tensors made
      only of tie values and compared with the CPU. On torch 2.10 / ROCm 7 it
      rounded the exact product once on its non-vectorised paths: every tie
      element of a tensor of at most 256 elements and of a misaligned view
      differed from the CPU by one unit, and so did the elements of an aligned
      tensor past its vectorised part (512 of 2,560); the vectorised part
      rounded twice like the CPU. Those counts are printed, not asserted (they
      are the torch build's, not the library's); the test asserts only that
      where the two differ they are one unit apart, a difference of tie
      rounding. The reference's expressions run by ROCm torch therefore
      differ from the reference (run on CUDA) on such ties, which is why the
      long runs compare against the CPU/CUDA recipe."""
    from dizo_amd.table import ZOTable
    lr, seed = 9.15e-07, 4321
    ties = _fp16_tie_values(lr)
    assert len(ties) >= 1
    rng_ = np.random.default_rng(5)
    # the library: theta - lr * (g * z) with z the exported normals, 1M elements,
    # against torch on the CPU; a few hundred of its products are ties
    n = 1 << 20
    gen = torch.Generator().manual_seed(8)
    theta = (torch.randn(n, generator=gen) * 1e-4).to(torch.float16)
    t = theta.cuda()
    tab = ZOTable([t])
    z = tab.export_z(seed, 0).cpu()
    gz = (z.float() * np.float32(-51.03125)).to(torch.float16)
    exact = gz.double().numpy() * np.float64(np.float32(lr))
    lib_ties = int((exact.astype(np.float16).view(np.int16)
                    != (gz.float() * np.float32(lr)).to(torch.float16).numpy().view(np.int16)).sum())
    assert lib_ties >= 20, f"only {lib_ties} tie elements"
    tab.update(seed, -51.03125, lr)
    cpu = [theta.clone()]
    R.zo_update(cpu, [z], -51.03125, lr)
    torch.cuda.synchronize()
    assert torch.equal(t.cpu().view(torch.int16), cpu[0].view(torch.int16))
    tab.close()

    # ROCm torch's kernel on tensors made only of tie values; lr * c is applied
    # to c itself (a view when off > 0: g * c would hand it a fresh aligned copy)
    widest = 0

    def rocm_vs_cpu(n: int, off: int) -> int:
        nonlocal widest
        vals = torch.from_numpy(rng_.choice(np.concatenate([ties, -ties]), size=n + off).astype(np.float16))
        dev = vals.cuda()[off:]
        got = (lr * dev).cpu().view(torch.int16).long()
        want = (lr * vals[off:]).view(torch.int16).long()
        widest = max(widest, int((got - want).abs().max()))
        return int((got != want).sum())

    small = [rocm_vs_cpu(k, 0) for k in (1, 7, 64, 256)]
    misaligned = [rocm_vs_cpu(k, 1) for k in (2560, 65536)]
    tail = rocm_vs_cpu(2560, 0)
    body = rocm_vs_cpu(65536, 0)
    print(f"ROCm torch vs CPU on tie elements: n=1,7,64,256 -> {small}; misaligned 2560, 65536 -> {misaligned}; "
          f"aligned 2560 -> {tail}; aligned 65536 -> {body}", flush=True)
    assert widest <= 1, f"ROCm torch and the CPU differ by {widest} units on tie products"


@pytest.mark.parametrize("prefetch", [False, True])
def test_single_tensor_beyond_2_32_elements(prefetch):
    """One fp16 tensor of 2^32 + 8200 elements (8.6 GB), its z offset past 2^32
    as well: perturb and the fused restore+update+perturb (plain and
    prefetching tile loops), checked against the oracle on windows at the
    start, across the 2^32 element boundary and at the ragged end."""
    n = (1 << 32) + 8200
    t = torch.zeros(n, dtype=torch.float16, device="cuda")
    off = 3 << 31  # the tensor's first z index
    tab = _fused_table([t], prefetch, z_offsets=[off])
    seed, eps, g, lr = 99, 1e-3, -1.25, 1e-6
    tab.perturb(seed, 1.0, eps)
    tab.restore_update_perturb(seed, seed + 1, eps, g, lr)
    torch.cuda.synchronize()
    for start in (0, (1 << 32) - 4096, n - 5000):
        m = min(9000, n - start)
        z1 = rng.tensor_z_bits(seed, off + start, m, F16)
        z2 = rng.tensor_z_bits(seed + 1, off + start, m, F16)
        th = np.zeros(m, dtype=np.uint16)
        want = A.perturb(A.restore_update(A.perturb(th, z1, 1, eps, F16), z1, eps, g, lr, F16), z2, 1, eps, F16)
        got = t[start:start + m].cpu().view(torch.int16).numpy().view(np.uint16)
        assert np.array_equal(got, want), start
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("prefetch", [False, True, None])
def test_tiles_across_the_2_32_counter_boundary(dt, prefetch):
    """Philox counters q = e >> 3 past 2^32: z offsets put one tile of each tile
    size across q = 2^32 (its counters' high word changes inside the tile),
    the tiles before it at high word 0 and the tiles after it at high word 1.
    Every mode (perturb, update, restore+update, restore+update+next perturb;
    the last on the plain and the prefetching tile loop, which hands a tile
    across the boundary to the plain loop), every element against the oracle."""
    sizes = [200_000, 70_001]
    # the first tensor starts 5000 groups below q = 2^32; the second 904 groups
    # below q = 2^33, so its first tile crosses at once
    offs = [(1 << 35) - 8 * 5000, (1 << 36) - 8 * 904]
    host = [random_theta(n, dt, 40 + i) for i, n in enumerate(sizes)]
    dev = torch.device("cuda", 0)
    tensors = [to_torch(b, dt, dev) for b in host]
    tab = _fused_table(tensors, prefetch, z_offsets=offs)
    seed, seed2, eps, g, lr = 512, 513, 1e-3, 0.75, 1e-3
    z1 = [rng.tensor_z_bits(seed, o, n, dt) for o, n in zip(offs, sizes)]
    z2 = [rng.tensor_z_bits(seed2, o, n, dt) for o, n in zip(offs, sizes)]
    want = list(host)

    def check(what):
        torch.cuda.synchronize()
        for i, t in enumerate(tensors):
            assert_bits_equal(to_bits(t).ravel(), want[i], dt, f"{what}, tensor {i}")

    tab.perturb(seed, 1.0, eps)
    want = [A.perturb(w, z, 1, eps, dt) for w, z in zip(want, z1)]
    check("perturb")
    tab.update(seed, g, lr)
    want = [A.update(w, z, g, lr, dt) for w, z in zip(want, z1)]
    check("update")
    tab.restore_update(seed, eps, g, lr)
    want = [A.restore_update(w, z, eps, g, lr, dt) for w, z in zip(want, z1)]
    check("restore+update")
    tab.restore_update_perturb(seed, seed2, eps, g, lr)
    want = [A.perturb(A.restore_update(w, z, eps, g, lr, dt), zz, 1, eps, dt)
            for w, z, zz in zip(want, z1, z2)]
    check("restore+update+next perturb")
    tab.close()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("prefetch", [False, True, None])
def test_special_values_follow_ieee_like_the_oracle(dt, prefetch):
    """theta holding +-inf, NaN, +-0, the largest finite value and the smallest
    subnormal, among ordinary values: every RMW mode, then the projection's
    apply and reverse with a supplied alpha, against the oracle (NaN equal to
    NaN, as torch's expressions give NaN there too)."""
    from dizo_amd._lib import DZ_PROJ_APPLY, DZ_PROJ_REVERSE
    from dizo_amd.table import ProjTable
    big = {F16: 65504.0, BF16: 3.3895314e38, F32: 3.4028235e38}[dt]
    tiny = {F16: 5.96e-8, BF16: 9.2e-41, F32: 1.4e-45}[dt]
    specials = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, big, -big, tiny, -tiny], dtype=np.float32)
    n = 40_003
    x = (np.random.default_rng(5).standard_normal(n) * 0.02).astype(np.float32)
    x[::97] = np.resize(specials, x[::97].size)
    h0 = A.from_f32(x, dt)
    dev = torch.device("cuda", 0)
    t = to_torch(h0, dt, dev)
    tab = _fused_table([t], prefetch)
    seed, seed2, eps, g, lr = 77, 78, 1e-3, 2.5, 1e-3
    z = rng.tensor_z_bits(seed, 0, n, dt)
    z2 = rng.tensor_z_bits(seed2, 0, n, dt)
    want = A.perturb(h0, z, 1, eps, dt)
    tab.perturb(seed, 1.0, eps)
    assert_bits_equal(to_bits(t).ravel(), want, dt, "perturb")
    want = A.update(want, z, g, lr, dt)
    tab.update(seed, g, lr)
    assert_bits_equal(to_bits(t).ravel(), want, dt, "update")
    want = A.restore_update(want, z, eps, g, lr, dt)
    tab.restore_update(seed, eps, g, lr)
    assert_bits_equal(to_bits(t).ravel(), want, dt, "restore+update")
    want = A.perturb(A.restore_update(want, z, eps, g, lr, dt), z2, 1, eps, dt)
    tab.restore_update_perturb(seed, seed2, eps, g, lr)
    assert_bits_equal(to_bits(t).ravel(), want, dt, "restore+update+next perturb")
    tab.close()
    # projection: theta0 is the starting theta (finite where theta is, so
    # inf - theta0 = inf and NaN stays NaN)
    anchor = to_torch(h0, dt, dev)
    ptab = ProjTable([t], [anchor])
    alpha_bits = A.from_f32(np.float32(0.75), dt).reshape(1)
    alpha = to_torch(alpha_bits, dt, dev)
    ptab.project(alpha, DZ_PROJ_APPLY)
    want = A.apply(want, h0, alpha_bits, dt)
    assert_bits_equal(to_bits(t).ravel(), want, dt, "apply")
    ptab.project(alpha, DZ_PROJ_REVERSE)
    want = A.reverse(want, h0, alpha_bits, dt)
    assert_bits_equal(to_bits(t).ravel(), want, dt, "reverse")
    ptab.close()
