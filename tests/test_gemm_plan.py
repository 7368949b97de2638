"""How the batched product is cut into launches and where its waves read (qtip_gemm_plan.h), compiled for the host."""
import ctypes

import pytest

import gemm_plan as G
from gemm_plan import CUS, FEW, ROWS, SHARED, plan


@pytest.fixture(scope="module")
def native():
    return G.library()


def test_cases_reach_every_kernel():
    """The cases that the GPU runs reach the form they are listed for at every bit width, and between them every compiled one."""
    for m, k, rows, long_sums, form in G.FORMS + G.SHARED_FORMS:
        for bits in (3, 4) if form[:2] == (SHARED, 1) else (2, 3, 4):
            assert form in G.launches(m, k, bits, rows, not long_sums), (m, k, rows, bits)
    compiled = {(FEW, 1, 1), (FEW, 1, 2), (SHARED, 1, 2), (SHARED, 2, 2)} | {
        (ROWS, NB, RG) for NB, RG in ((8, 8), (8, 4), (6, 8), (4, 8), (4, 4), (4, 2), (2, 4), (2, 2))}
    reached = {(form[:3], form[4]) for *_, form in G.FORMS + G.SHARED_FORMS}
    assert reached == {(f, inside) for f in compiled for inside in (False, True)}
    assert any(G.plan(m, k, 2, rows, fine=False)[0] < m for m, k, rows, long_sums, _ in G.FORMS if long_sums)  # two launches


@pytest.mark.parametrize("k", [32, 64, 96, 832, 928, 2080, 4096, 28672])
@pytest.mark.parametrize("m", [32, 1056, 4096, 22016])
def test_few_rows_read_their_activations_only(native, m, k):
    """Every load of activations that gemm_few_kernel issues (the first whether or not the wave has a wave-load, then one for
    each) lies inside the batch, or has a lane offset out of range by itself and a scalar offset inside."""
    place = (ctypes.c_uint32 * 2)()
    nwl, odd = (k // 32 + 1) // 2, k // 32 % 2
    for batch in (2, 5, 16):
        _, (form, _, RG, S, wl_per), _ = plan(m, k, 2, batch)
        assert form == FEW
        KS, size = 16 // RG, batch * k * 2
        for s in sorted({0, S - 1}):
            wl1 = min((s + 1) * wl_per, nwl)
            for ks in range(KS):
                first = s * wl_per + ks
                nst = max(0, -(-(wl1 - first) // KS))
                half = bool(odd and nst and first + KS * (nst - 1) == nwl - 1)
                for units in (1, 0):
                    for lane in range(64):
                        native.few_place(lane, batch, k, first, units, nst, int(half), place)
                        so, vo = place
                        for t in range(nst if units and nst else 1):
                            last = half and t == nst - 1 and lane >= 32  # (the kernel takes these lanes out of range)
                            assert so <= size
                            if vo < 0x7FFFFF00 and not (last and t):
                                assert so + vo + 32 + 16 <= size, (batch, s, ks, lane, t)
                            so += KS * 128


def _error(nwl, KS, wl_per, S):
    """Chains of additions on the matrix cores (which weigh 5), slices (1.5) and ranges (1) of a sum over nwl 64-column pieces."""
    n = min(wl_per, nwl)
    return 10 * -(-n // KS) + min(KS, n) * 3 // 2 + S


def _cut_error(m, k, batch, split):
    """_error of the cut that bounds it: passes of 128 rows in 8, 4 or 2 slices and ranges of 1024 or 512 columns."""
    if batch > 128:
        return min(_cut_error(m, k, 128, split), _cut_error(m, k, batch - 128, split))
    KS, RG, least = (8, 2, 16) if batch <= 32 else (4, 2, 8) if batch <= 64 else (2, 4, 8)
    nwl, groups = (k // 32 + 1) // 2, -(-((m // 32 + 1) // 2) // RG)
    S = 1
    while split and S < 16 and groups * S * 2 <= CUS and nwl // (2 * S) >= least:
        S *= 2
    wl_per = -(-(-(-nwl // S)) // KS) * KS
    return _error(nwl, KS, wl_per, -(-nwl // wl_per))


@pytest.mark.parametrize("k", [32, 96, 512, 832, 1120, 2048, 3328, 4096, 5504, 8192, 11008, 28672, 1 << 20, 1 << 23])
def test_sums_are_cut_finely(native, k):
    """Every pass of a product: chains, slices and ranges no coarser than the bound, with scratch for ranges and without."""
    nwl = (k // 32 + 1) // 2
    for m in (32, 96, 512, 992, 1728, 2048, 4096, 6144, 8192, 10240, 11008, 14336, 22016, 28672, 57344):
        for bits in (2, 4):
            for batch in (1, 2, 5, 9, 16, 17, 20, 32, 33, 48, 64, 65, 100, 128, 129, 150, 190, 256, 1000):
                for split in (True, False):
                    left = batch
                    while left:
                        nb = native.pass_of(m, k, bits, left, CUS, int(split), 1)
                        assert 1 <= nb <= min(left, 256) and nb * k * 2 <= 0x7FFFFF00
                        m0, (form, NB, RG, S, wl_per), _ = plan(m, k, bits, nb, split)
                        assert m0 == m and RG and (split or S == 1)
                        KS = (8 if form == ROWS else 16) // RG
                        assert _error(nwl, KS, wl_per, S) <= _cut_error(m, k, nb, split), (m, bits, batch, nb, split)
                        left -= nb


def test_long_sums_are_longer(native):
    _, (form, NB, RG, S, wl_per), _ = plan(8192, 28672, 2, 1000, fine=False)
    assert form == ROWS and _error(448, 8 // RG, wl_per, S) > 2 * _cut_error(8192, 28672, 128, True)


def test_sizes_that_share_a_slot_of_held_plans_part_again(native):
    """The plans of a thread's last sizes are held in 64 slots: no two projections share one at more than a sixteenth of the row
    counts (a sixty-fourth by chance), and a plan asked for again is the same after others have taken its slot."""
    sizes = [(m, k) for d, f, kv in ((4096, 11008, 4096), (2048, 5504, 512), (8192, 28672, 1024), (5120, 13824, 5120))
             for m, k in ((d, d), (kv, d), (f, d), (2 * f, d), (d, f))] + [(m, k) for m in (832, 928, 1120) for k in (832, 928, 1120)]
    slots = {s: [native.slot_of(*s, bits, nb, 1, 1) for nb in range(1, 513) for bits in (2, 4)] for s in set(sizes)}
    assert all(0 <= v < 64 for l in slots.values() for v in l)
    for a in slots:
        for b in slots:
            assert a == b or sum(x == y for x, y in zip(slots[a], slots[b])) <= 1024 // 16, (a, b)
    cases = [(m, k, bits, nb, split, fine) for m, k in sizes for bits in (2, 3) for nb in (5, 40, 300) for split in (0, 1) for fine in (0, 1)]
    first = [plan(*c) for c in cases]
    assert [plan(*c) for c in reversed(cases)] == first[::-1]
