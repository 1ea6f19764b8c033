"""GPU parity of the standalone merge (moba_hip_merge, the counterpart of
merge_forward in src/moba_opt/ops/bindings.cpp:6-22) against the FP64 oracle
merge (reference/merge_reference.py:10-26), including the reference's own
cases (tests/test_merge_cuda.py:27-31: no remote rows is the identity) and
the closed-form edge cases pinned on the oracle in tests/test_oracle.py."""
import numpy as np
import pytest
import torch

from helpers import assert_close_stats
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(T, H, D, dtype, per_row_max, seed, shuffle=True):
    g = torch.Generator().manual_seed(seed)
    rng = np.random.default_rng(seed)
    so = torch.randn((T, H, D), generator=g)
    sl = torch.randn((T, H), generator=g) * 3
    counts = rng.integers(0, per_row_max + 1, T * H)
    mapping = np.repeat(np.arange(T * H), counts)
    if shuffle:
        rng.shuffle(mapping)
    M = len(mapping)
    ro = torch.randn((M, D), generator=g)
    rl = torch.randn(M, generator=g) * 3
    dev = "cuda"
    return (so.to(dev, dtype), sl.to(dev), ro.to(dev, dtype), rl.to(dev),
            torch.from_numpy(mapping).to(dev))


def _ref(so, sl, ro, rl, mp):
    T, H, D = so.shape
    o, l = O.merge(so.double().cpu().numpy().reshape(T * H, D), sl.double().cpu().numpy().reshape(-1),
                   ro.double().cpu().numpy(), rl.double().cpu().numpy(), mp.cpu().numpy())
    return o.reshape(T, H, D), l.reshape(T, H)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,D,per_row", [(37, 5, 64, 3), (9, 4, 8, 8), (50, 2, 96, 1),
                                           (11, 3, 256, 5)])
def test_merge_matches_fp64(cuda_device, T, H, D, per_row, dtype):
    from moba_hip.merge import merge_forward
    so, sl, ro, rl, mp = _case(T, H, D, dtype, per_row, seed=T * 7 + D)
    out, lse = merge_forward(so, sl, ro, rl, mp)
    o_ref, l_ref = _ref(so, sl, ro, rl, mp)
    assert out.dtype == dtype and lse.dtype == torch.float32
    if dtype == torch.float32:
        np.testing.assert_allclose(out.double().cpu().numpy(), o_ref, atol=2e-6, rtol=1e-5)
    else:
        assert_close_stats(out, o_ref, dtype, "merged out")
    np.testing.assert_allclose(lse.double().cpu().numpy(), l_ref, atol=2e-6, rtol=1e-6)
    again = merge_forward(so, sl, ro, rl, mp)
    assert torch.equal(out, again[0]) and torch.equal(lse, again[1])


@pytest.mark.parametrize("T,H", [(4096, 8), (70000, 1)])
def test_merge_multi_pass_sort(cuda_device, T, H):
    """P = 32768 (two 8-bit digit passes) and P = 70000 (three), with up to
    7 remote partials per row in shuffled order."""
    from moba_hip.merge import merge_forward
    so, sl, ro, rl, mp = _case(T, H, 64, torch.bfloat16, 7, seed=T)
    out, lse = merge_forward(so, sl, ro, rl, mp, kmax=7)
    o_ref, l_ref = _ref(so, sl, ro, rl, mp)
    assert_close_stats(out, o_ref, torch.bfloat16, "merged out")
    np.testing.assert_allclose(lse.double().cpu().numpy(), l_ref, atol=2e-6, rtol=1e-6)


def test_merge_no_remote_is_identity(cuda_device):
    from moba_hip.merge import merge_forward
    so, sl, _, _, _ = _case(6, 3, 32, torch.bfloat16, 0, seed=3)
    ro = torch.empty((0, 32), device="cuda", dtype=torch.bfloat16)
    rl = torch.empty(0, device="cuda")
    mp = torch.empty(0, device="cuda", dtype=torch.int64)
    out, lse = merge_forward(so, sl, ro, rl, mp)
    assert torch.equal(out, so) and torch.equal(lse, sl)


def test_merge_extreme_lse_gap(cuda_device):
    from moba_hip.merge import merge_forward
    so, sl, ro, rl, _ = _case(5, 1, 16, torch.float32, 0, seed=4)
    ro = torch.randn((5, 16), device="cuda")
    mp = torch.arange(5, device="cuda")
    out, lse = merge_forward(so, torch.full_like(sl, -1e30), ro, torch.full((5,), 1e30,
                             device="cuda"), mp)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
    torch.testing.assert_close(out[:, 0], ro, atol=1e-6, rtol=0)


def test_merge_capacity_and_range_errors(cuda_device):
    from moba_hip.merge import merge_forward
    so, sl, ro, rl, _ = _case(4, 2, 16, torch.bfloat16, 0, seed=5)
    ro = torch.randn((5, 16), device="cuda").bfloat16()
    rl = torch.randn(5, device="cuda")
    crowded = torch.tensor([3, 3, 3, 1, 0], device="cuda")
    with pytest.raises(RuntimeError, match="capacity exceeded"):
        merge_forward(so, sl, ro, rl, crowded, kmax=2)
    merge_forward(so, sl, ro, rl, crowded, kmax=2, check_capacity=False)  # no raise
    with pytest.raises(RuntimeError, match=r"\[0,T\*H\)"):
        merge_forward(so, sl, ro, rl, torch.tensor([0, 1, 8, 2, 3], device="cuda"))
    # negative and far-out entries with the derived kmax reach the same native check
    for bad in ([0, -1, 2, 3, 4], [0, 1, 2, 3, 1 << 40], [-5, -5, -5, -5, -5]):
        with pytest.raises(RuntimeError, match=r"\[0,T\*H\)"):
            merge_forward(so, sl, ro, rl, torch.tensor(bad, device="cuda"))
    with pytest.raises(ValueError, match="deterministic"):
        merge_forward(so, sl, ro, rl, crowded, deterministic=1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kmax,counts", [(1, (2, 0, 1)), (3, (5, 3, 0, 4)), (4, (9, 4)),
                                         (8, (300, 8, 1))])
def test_merge_keeps_the_first_kmax_partials(cuda_device, kmax, counts, dtype):
    """Rows with fewer, exactly and more remote partials than kmax (up to a
    row that a whole workgroup of partials meets in): each keeps its kmax
    lowest indices, in every run, for int32 and int64 mappings, and for inputs
    whose rows do not start on 16 bytes."""
    from moba_hip.merge import merge_forward
    g = torch.Generator().manual_seed(kmax)
    n, D = len(counts), 40
    mapping = np.repeat(np.arange(n), counts)
    np.random.default_rng(kmax).shuffle(mapping)
    M = len(mapping)
    step = 4 if dtype == torch.float32 else 2

    def shifted(*shape):   # contiguous, `step * 2` bytes past an aligned start
        flat = torch.randn(int(np.prod(shape)) + 16, generator=g).to("cuda", dtype)
        return flat[8 // step:8 // step + int(np.prod(shape))].view(*shape)
    so, ro = shifted(n, 1, D), shifted(M, D)
    sl, rl = torch.randn(n, 1, generator=g).cuda(), torch.randn(M, generator=g).cuda()
    keep = np.concatenate([np.flatnonzero(mapping == r)[:kmax] for r in range(n)]).astype(int)
    ref = _ref(so, sl, ro[keep], rl[keep], torch.from_numpy(mapping[keep]))
    first = None
    for mp in (torch.from_numpy(mapping).cuda(), torch.from_numpy(mapping).int().cuda()):
        for _ in range(3):
            out, lse = merge_forward(so, sl, ro, rl, mp, kmax=kmax, check_capacity=False)
            first = first or (out, lse)
            assert torch.equal(out, first[0]) and torch.equal(lse, first[1])
    if dtype == torch.float32:
        np.testing.assert_allclose(out.double().cpu().numpy(), ref[0], atol=2e-6, rtol=1e-5)
    else:
        assert_close_stats(out, ref[0], dtype, "merged out")
    np.testing.assert_allclose(lse.double().cpu().numpy(), ref[1], atol=2e-6, rtol=1e-6)
    with pytest.raises(RuntimeError, match="capacity exceeded"):
        merge_forward(so, sl, ro, rl, mp, kmax=kmax)


@pytest.mark.parametrize("kmax", [1, 2, 8])
@pytest.mark.parametrize("rows", ["one", "two in turn", "sixteen in turn", "runs of ten",
                                  "one among many"])
def test_merge_of_crowded_rows(cuda_device, rows, kmax):
    """Mappings in which waves meet in a few rows: the first kmax partials of
    each row are merged, and the call takes no more than ten times one whose
    partials are spread out (minima on one address are served one by one: 400
    times, when every partial took them)."""
    from moba_hip.merge import merge_forward
    g = torch.Generator().manual_seed(kmax)
    T, H, D, M = 4096, 2, 64, 100_003
    j = np.arange(M)
    mapping = {"one": np.full(M, 777), "two in turn": j % 2 * 256, "sixteen in turn": j % 16 * 100,
               "runs of ten": j // 10 % (T * H),
               "one among many": np.where(j % 3 == 0, 4097, j % (T * H))}[rows]
    so, ro = torch.randn(T, H, D, generator=g).cuda(), torch.randn(M, D, generator=g).cuda()
    sl, rl = torch.randn(T, H, generator=g).cuda(), torch.randn(M, generator=g).cuda()

    def call(m):
        m = torch.from_numpy(m).int().cuda()
        best = []
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            out = merge_forward(so, sl, ro, rl, m, kmax=kmax, check_capacity=False)
            b.record()
            torch.cuda.synchronize()
            best.append(a.elapsed_time(b))
        return out, min(best)
    (out, lse), took = call(mapping)
    order = np.argsort(mapping, kind="stable")
    start = np.searchsorted(mapping[order], mapping[order], "left")
    keep = np.sort(order[np.arange(M) - start < kmax])
    ref = _ref(so, sl, ro[keep], rl[keep], torch.from_numpy(mapping[keep]))
    np.testing.assert_allclose(out.double().cpu().numpy(), ref[0], atol=2e-6, rtol=1e-5)
    np.testing.assert_allclose(lse.double().cpu().numpy(), ref[1], atol=2e-6, rtol=1e-6)
    _, spread = call(np.random.default_rng(0).permutation(M) % (T * H))
    assert took <= 10 * spread, f"{took * 1e3:.0f} us against {spread * 1e3:.0f}"
