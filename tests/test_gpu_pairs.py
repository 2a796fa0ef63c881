"""
GPU checks of the structured path (merged pair- and single-excitation coefficients applied by the
core-group gather kernels, the diagonal kernel, and the remaining terms on the enumeration kernel)
against the oracle and against the enumeration-only path:

  - forward through the pair path equals oracle apply_within within 1e-12 relative to each entry's
    sum of |contributions|, for molecular tables (Hermitian, pc = 1), random non-Hermitian tables
    over two config words (pc = 1 and 2) and every symmetric setting;
  - the adjoint through the pair path equals the enumeration-only adjoint (itself checked against
    the dense conjugate transpose elsewhere);
  - the split is exact: every valid term lands in exactly one of the pair table, the single table,
    the diagonal records or the residual enumeration;
  - the pair path is refused for foreign config sets and chosen automatically otherwise.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import sorted_terms
from oracle import oracle as orc
from qmb_hip import _lib
from qmb_hip import autograd as ag
from qmb_hip import prepared as pp
from qmb_hip import synthetic as sy

pytestmark = pytest.mark.gpu


def _pair_heavy_table(sites: np.ndarray, n_terms: int, seed: int) -> tuple[np.ndarray, np.ndarray, np.ndarray]:
    """Random non-Hermitian table on `sites`: pair excitations in every operator order, hops,
    number-dressed hops and diagonal terms."""
    rng = np.random.default_rng(seed)
    site = np.zeros((n_terms, 4), dtype=np.int16)
    kind = np.full((n_terms, 4), 2, dtype=np.uint8)
    for t in range(n_terms):
        u = rng.random()
        if u < 0.5:  # pair excitation, any operator order
            site[t] = rng.choice(sites, size=4, replace=False)
            kind[t] = rng.permutation([0, 0, 1, 1])
        elif u < 0.65:  # hop
            site[t, :2] = rng.choice(sites, size=2, replace=False)
            kind[t, :2] = [1, 0]
        elif u < 0.75:  # hop dressed by an occupied site: a+_p a+_k a_k a_r
            p, k, r = rng.choice(sites, size=3, replace=False)
            site[t] = [p, k, k, r]
            kind[t] = [1, 1, 0, 0]
        elif u < 0.82:  # hop dressed by an empty site: a+_p a_k a+_k a_r
            p, k, r = rng.choice(sites, size=3, replace=False)
            site[t] = [p, k, k, r]
            kind[t] = [1, 0, 1, 0]
        elif u < 0.9:  # diagonal: n_p or n_p n_q
            p, q = rng.choice(sites, size=2, replace=False)
            if rng.random() < 0.5:
                site[t, :2] = [p, p]
                kind[t, :2] = [1, 0]
            else:
                site[t] = [p, q, q, p]
                kind[t] = [1, 1, 0, 0]
        else:  # neither: a+_p a+_q a_r (changes the particle number)
            site[t, :3] = rng.choice(sites, size=3, replace=False)
            kind[t, :3] = [1, 1, 0]
    coef = rng.normal(size=(n_terms, 2))
    return site, kind, coef


def _fixed_weight_configs(sites: np.ndarray, weight: int, nq: int) -> np.ndarray:
    from itertools import combinations  # pylint: disable=import-outside-toplevel

    rows = []
    for comb in combinations(sites.tolist(), weight):
        bits = np.zeros(8 * nq, dtype=np.uint8)
        bits[list(comb)] = 1
        rows.append(np.packbits(bits, bitorder="little"))
    return sy.sort_unique_configs(np.array(rows, dtype=np.uint8))


def _two_word_case(pc: int) -> tuple[tuple[np.ndarray, np.ndarray, np.ndarray], np.ndarray]:
    sites = np.array([0, 1, 2, 3, 5, 8, 13, 30, 63, 64, 65, 66, 70, 71], dtype=np.int64)  # both words of nq = 9
    return _pair_heavy_table(sites, 900, 40 + pc), _fixed_weight_configs(sites, 5, 9)


CASES = [
    ("molecular-20so", 1, lambda: (sorted_terms(*sy.molecular_terms(10, 1001)), sy.sector_configs(10, 5, 5, 3000, 2))),
    ("molecular-8so-full-sector", 1, lambda: (sorted_terms(*sy.molecular_terms(4, 3)), sy.sector_configs(4, 2, 2, 36, 0))),
    ("random-two-words-fermi", 1, lambda: _two_word_case(1)),
    ("random-two-words-bose2", 2, lambda: _two_word_case(2)),
]


def _compile(site4: np.ndarray, kind4: np.ndarray, pc: int, nq: int) -> tuple[int, int]:
    lib = _lib.library()
    s = np.ascontiguousarray(site4, dtype=np.int16)
    k = np.ascontiguousarray(kind4, dtype=np.uint8)
    rec, status, bucket, diag = ctypes.c_uint64(0), ctypes.c_int32(0), ctypes.c_int64(0), ctypes.c_int32(0)
    _lib.check(lib.qmb_compile_term_host(s.ctypes.data, k.ctypes.data, pc, nq, ctypes.byref(rec), ctypes.byref(status),
                                         ctypes.byref(bucket), ctypes.byref(diag)), "compile")
    return rec.value, status.value


def _dev(x: np.ndarray, device: torch.device) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


@pytest.mark.parametrize("name,pc,case_fn", CASES, ids=[c[0] for c in CASES])
def test_pair_path_forward_matches_oracle(cuda_device: torch.device, name: str, pc: int, case_fn: object) -> None:
    (s, k, c), cfg = case_fn()
    nq = cfg.shape[1]
    psi = sy.random_psi(len(cfg), 17)
    want, asum, _ = orc.apply_within(pc, cfg, psi, cfg, s, k, c)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, pc)
    assert terms.pairs_desc is not None and terms.n_pair_terms > 0
    cfg_t = _dev(cfg, cuda_device)
    targets = pp.PreparedTargets(cfg_t, nq)
    assert pp.can_use_pairs(terms, targets, cfg_t)
    vec = torch.view_as_real(_dev(psi, cuda_device)).contiguous()
    settings = [pp.SYMMETRIC_OFF] + ([pp.SYMMETRIC_GATHER, pp.SYMMETRIC_HALF] if terms.hermitian else [])
    for symmetric in settings:
        for strategy in (pp.STRATEGY_TILES, pp.STRATEGY_DIRECT):
            out = pp.apply(terms, targets, cfg_t, vec, pp.MODE_FORWARD, strategy=strategy, symmetric=symmetric, pairs=True)
            got = out[:, 0].cpu().numpy() + 1j * out[:, 1].cpu().numpy()
            err = np.abs(got - want)
            assert np.all(err <= 1e-12 * asum + 1e-300), (name, symmetric, strategy, err.max())


@pytest.mark.parametrize("name,pc,case_fn", CASES, ids=[c[0] for c in CASES])
def test_pair_path_adjoint_matches_enumeration(cuda_device: torch.device, name: str, pc: int, case_fn: object) -> None:
    (s, k, c), cfg = case_fn()
    nq = cfg.shape[1]
    g = sy.random_psi(len(cfg), 23)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, pc)
    cfg_t = _dev(cfg, cuda_device)
    targets = pp.PreparedTargets(cfg_t, nq)
    vec = torch.view_as_real(_dev(g, cuda_device)).contiguous()
    ref = pp.apply(terms, targets, cfg_t, vec, pp.MODE_ADJOINT, symmetric=False, pairs=False).cpu().numpy()
    # the scale of each entry: the adjoint of |A| applied to |g|
    absmax = np.abs(c).sum(axis=1).max()
    scale = np.abs(ref).sum(axis=1) + absmax * np.abs(g).sum()
    for symmetric in ([pp.SYMMETRIC_OFF, pp.SYMMETRIC_GATHER] if terms.hermitian else [pp.SYMMETRIC_OFF]):
        got = pp.apply(terms, targets, cfg_t, vec, pp.MODE_ADJOINT, symmetric=symmetric, pairs=True).cpu().numpy()
        err = np.abs(got - ref).max(axis=1)
        assert np.all(err <= 1e-12 * scale), (name, symmetric, err.max())


@pytest.mark.parametrize("name,pc,case_fn", CASES, ids=[c[0] for c in CASES])
def test_structured_split_is_exact(cuda_device: torch.device, name: str, pc: int, case_fn: object) -> None:
    """Every valid term goes to exactly one of: pair table, single table, diagonal records, residual
    enumeration; the device counts agree with the host classifiers."""
    (s, k, c), cfg = case_fn()
    nq = cfg.shape[1]
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, pc)
    full_valid, full_diag, _ = terms.counts()
    assert terms.n_residual_terms + terms.n_pair_terms + terms.n_single_terms + full_diag == full_valid, name
    off = int(terms.pairs_desc.counts) - terms.pairs_buffer.data_ptr()
    assert int(terms.pairs_buffer[off + 8:off + 16].view(torch.int64).item()) == full_diag  # every diagonal term folded
    # real tables switch the pair kernels to 8-byte coefficients, and no merged entry has an imaginary part
    assert terms.pairs_desc.real == int(np.all(np.asarray(c)[:, 1] == 0)), name
    if terms.pairs_desc.real:
        assert int(terms.pairs_buffer[off + 16:off + 24].view(torch.int64).item()) == 0
    lib = _lib.library()
    out = (ctypes.c_int32 * 5)()
    n_pairs = n_singles = 0
    for row_s, row_k in zip(s, k):
        rec, status = _compile(row_s, row_k, pc, nq)
        if status != 0:
            continue
        n_pairs += lib.qmb_pair_excitation_host(rec, pc, out)
        n_singles += lib.qmb_single_excitation_host(rec, pc, out)
    assert (n_pairs, n_singles) == (terms.n_pair_terms, terms.n_single_terms), name
    if name.startswith("molecular"):
        assert terms.n_residual_terms == 0  # one-body, two-body and constant terms are all structured


def test_pair_path_selection(cuda_device: torch.device) -> None:
    s, k, c = sorted_terms(*sy.molecular_terms(4, 3))
    cfg = sy.sector_configs(4, 2, 2, 36, 0)
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), 1, 1)
    targets = pp.PreparedTargets(cfg_t, 1)
    assert pp.can_use_pairs(terms, targets, cfg_t)
    assert not pp.can_use_pairs(terms, targets, cfg_t.clone())
    vec = torch.view_as_real(_dev(sy.random_psi(36, 3), cuda_device)).contiguous()
    with pytest.raises(RuntimeError):
        pp.apply(terms, targets, cfg_t.clone(), vec, pp.MODE_FORWARD, pairs=True)
    no_pairs = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), 1, 1, pairs=False)
    assert no_pairs.pairs_desc is None and not pp.can_use_pairs(no_pairs, targets, cfg_t)
    # energy gradient through autograd takes the pair path and matches the enumeration-only terms
    psi = _dev(sy.random_psi(36, 5), cuda_device)
    grads = []
    for t in (terms, no_pairs):
        x = psi.clone().requires_grad_(True)
        ag.energy(x, cfg_t, t, targets).backward()
        grads.append(x.grad.cpu().numpy())
    np.testing.assert_allclose(grads[0], grads[1], atol=1e-12)


ACROSS = ["disjoint", "subset", "superset", "overlap", "repeated-source-rows", "repeated-missing-rows", "repeated-target-rows"]


@pytest.mark.parametrize("case", ACROSS)
def test_apply_across_matches_oracle(cuda_device: torch.device, case: str) -> None:
    """The structured path between two config sets (one joint set holding both) against the oracle,
    forward and adjoint; a target set with repeated rows is left to the enumeration kernel."""
    s, k, c = sorted_terms(*sy.molecular_terms(10, 1001))
    pool = sy.sector_configs(10, 5, 5, 3000, 51)
    rng = np.random.default_rng(52)
    perm = rng.permutation(len(pool))
    a, b = pool[perm[:1200]], pool[perm[1200:2400]]
    cfg_i, cfg_j = {
        "disjoint": (a, b),
        "subset": (a[:500], a),
        "superset": (a, a[:500]),
        "overlap": (np.concatenate([a[:700], b[:300]]), np.concatenate([a[400:900], b[200:900]])),
        "repeated-source-rows": (np.concatenate([a[:600], a[:100]]), a),  # repeats that configs_j holds: inputs add up
        "repeated-missing-rows": (np.concatenate([a, a[:100]]), b),  # repeats that configs_j lacks: not covered
        "repeated-target-rows": (a, np.concatenate([b, b[:50]])),
    }[case]
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), 3, 1)
    psi = sy.random_psi(len(cfg_i), 53)
    g = sy.random_psi(len(cfg_j), 54)
    ci, cj = _dev(cfg_i, cuda_device), _dev(cfg_j, cuda_device)
    fwd = pp.apply_across(terms, ci, torch.view_as_real(_dev(psi, cuda_device)).contiguous(), cj, pp.MODE_FORWARD)
    adj = pp.apply_across(terms, ci, torch.view_as_real(_dev(g, cuda_device)).contiguous(), cj, pp.MODE_ADJOINT)
    if case in ("repeated-target-rows", "repeated-missing-rows"):
        assert fwd is None and adj is None
        return
    want, asum, _ = orc.apply_within(1, cfg_i, psi, cfg_j, s, k, c)
    got = fwd.cpu().numpy()
    assert np.all(np.abs(got[:, 0] + 1j * got[:, 1] - want) <= 1e-12 * asum + 1e-300), case
    # adjoint: <g, A psi> = <A^H g, psi> for every psi, so compare with the dense columns' conjugate sums
    ref = pp.apply(terms, pp.PreparedTargets(cj, 3), ci, torch.view_as_real(_dev(g, cuda_device)).contiguous(), pp.MODE_ADJOINT,
                   pairs=False).cpu().numpy()
    got_a = adj.cpu().numpy()
    scale = np.abs(ref).sum(axis=1) + np.abs(c).sum(axis=1).max() * np.abs(g).sum()
    assert np.all(np.abs(got_a - ref).max(axis=1) <= 1e-12 * scale), case


def test_too_low_max_occupied_raises(cuda_device: torch.device) -> None:
    """A max_occupied bound below a row's occupancy is an error from the core index build, not a
    NaN row or missing pair terms."""
    s, k, c = sorted_terms(*sy.molecular_terms(6, 21))
    cfg = torch.from_numpy(sy.sector_configs(6, 3, 3, 120, 22)).to(cuda_device)
    terms = pp.PreparedTerms(torch.from_numpy(s).to(cuda_device), torch.from_numpy(k).to(cuda_device),
                             torch.from_numpy(c).to(cuda_device), 2, 1)
    vec = torch.zeros((cfg.size(0), 2), dtype=torch.float64, device=cuda_device)
    low = pp.PreparedTargets(cfg, 2, distinct=True, max_occupied=5)
    with pytest.raises(RuntimeError, match="max_occupied=5"):
        pp.apply(terms, low, cfg, vec, pp.MODE_FORWARD)
    exact = pp.PreparedTargets(cfg, 2, distinct=True, max_occupied=6)
    assert torch.isfinite(pp.apply(terms, exact, cfg, vec, pp.MODE_FORWARD)).all()


def _core_index(targets: pp.PreparedTargets, order: int) -> tuple[np.ndarray, np.ndarray, np.ndarray]:
    """(vals, starts with their flag bit, counts) of a built core index, copied to the host."""
    desc = targets.cores(order)
    buf = targets._cores[order][0]  # pylint: disable=protected-access
    base = buf.data_ptr()
    counts = buf[int(desc.counts) - base:int(desc.counts) - base + 32].view(torch.int64).cpu().numpy()
    entries, groups = int(counts[0]), int(counts[1])
    vals = buf[int(desc.vals) - base:int(desc.vals) - base + 8 * entries].view(torch.int64).cpu().numpy().astype(np.uint64)
    off = int(desc.starts) - base
    starts = buf[off:off + 4 * (groups + 1)].view(torch.int32).cpu().numpy().astype(np.uint32)
    return vals, starts, counts


def _build_cores_with_narrow_hash(targets: pp.PreparedTargets, bits: int, seed: int) -> None:
    """Builds both core indexes of the set from random `bits`-bit hash columns, so that many
    different cores share a key, then puts the set's own columns back (its hash index, built later
    on first use, keeps them)."""
    off = int(targets.keys_desc.cols) - targets.buffer.data_ptr()
    view = targets.buffer[off:off + 8 * 256].view(torch.int64)
    own = view.clone()
    rng = np.random.default_rng(seed)
    view.copy_(torch.from_numpy(rng.integers(0, 1 << bits, size=256, dtype=np.int64)))
    targets.cores(2)
    targets.cores(1)
    view.copy_(own)


MERGE_CASES = [c for c in CASES if c[0] in ("molecular-20so", "random-two-words-fermi")]


@pytest.mark.parametrize("bits", [3, 9, 12, 14])
@pytest.mark.parametrize("name,pc,case_fn", MERGE_CASES, ids=[c[0] for c in MERGE_CASES])
def test_merged_core_groups(cuda_device: torch.device, name: str, pc: int, case_fn: object, bits: int) -> None:
    """Core keys from narrowed hash columns merge many different cores into one group (3 bits: a
    few thousand entries a group; 14 bits: a few).  The build flags exactly the groups holding more
    than one core, and the forward and adjoint through those mixed groups -- every group class:
    2..8 entries, 9..32 packed, larger -- still equal the oracle and the enumeration."""
    (s, k, c), cfg = case_fn()
    nq = cfg.shape[1]
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, pc)
    targets = pp.PreparedTargets(cfg_t, nq, distinct=True)
    _build_cores_with_narrow_hash(targets, bits, 7 + bits)
    bitsof = np.unpackbits(cfg, axis=1, bitorder="little")
    sizes_seen = set()
    n_mixed = 0
    for order in (2, 1):
        vals, starts, _ = _core_index(targets, order)
        flag = starts[:-1] >> 31
        st = (starts & 0x7FFFFFFF).astype(np.int64)
        sizes = np.diff(st)
        assert st[0] == 0 and st[-1] == len(vals) and (sizes > 0).all()
        # the core of every entry: its row's sites without the removed ones
        rows = (vals >> np.uint64(16)).astype(np.int64)
        core = bitsof[rows].copy()
        e = np.arange(len(vals))
        core[e, (vals & np.uint64(0xFF)).astype(np.int64)] = 0
        if order == 2:
            core[e, ((vals >> np.uint64(8)) & np.uint64(0xFF)).astype(np.int64)] = 0
        packed = np.packbits(core, axis=1, bitorder="little")
        first = np.repeat(st[:-1], sizes)
        differs = (packed != packed[first]).any(axis=1).astype(np.int64)
        mixed = np.add.reduceat(differs, st[:-1]) > 0
        np.testing.assert_array_equal(flag.astype(bool), mixed)
        n_mixed += int(mixed.sum())
        sizes_seen.update(np.unique(np.minimum(sizes[mixed], 33)).tolist())
    if name.startswith("molecular"):
        # ~40k distinct cores: merged at every width, down to groups of 2..4 entries at 14 bits
        assert n_mixed > 0
        if bits == 14:
            assert {2, 3, 4}.issubset(sizes_seen), sizes_seen
    elif bits <= 9:
        assert n_mixed > 0  # a few hundred distinct cores merge only under narrow keys
    psi = sy.random_psi(len(cfg), 61)
    vec = torch.view_as_real(_dev(psi, cuda_device)).contiguous()
    want, asum, _ = orc.apply_within(pc, cfg, psi, cfg, s, k, c)
    got = pp.apply(terms, targets, cfg_t, vec, pp.MODE_FORWARD, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    err = np.abs(got[:, 0] + 1j * got[:, 1] - want)
    assert np.all(err <= 1e-12 * asum + 1e-300), (name, bits, err.max())
    ref = pp.apply(terms, pp.PreparedTargets(cfg_t, nq), cfg_t, vec, pp.MODE_ADJOINT, symmetric=False, pairs=False).cpu().numpy()
    got_a = pp.apply(terms, targets, cfg_t, vec, pp.MODE_ADJOINT, symmetric=False, pairs=True).cpu().numpy()
    scale = np.abs(ref).sum(axis=1) + np.abs(c).sum(axis=1).max() * np.abs(psi).sum()
    assert np.all(np.abs(got_a - ref).max(axis=1) <= 1e-12 * scale), (name, bits)



@pytest.mark.parametrize("bits", [0, 4])
@pytest.mark.parametrize("n", [1, 2, 60, 182, 183, 1000, 3000])
def test_core_index_builds_around_the_one_block_limit(cuda_device: torch.device, n: int, bits: int) -> None:
    """Sets of 10 electrons (45 entries a row) on both sides of the 8192 entries that one block indexes
    (182 rows: 8190) and of the radix sort's lower limit (1000 rows: 45,000; 3000: 135,000), with the
    set's hash and with 4-bit hash columns (nearly every group mixed): the sorted index equals one
    made on the host, and both modes equal the oracle and the enumeration."""
    s, k, c = sorted_terms(*sy.molecular_terms(10, 31))
    cfg = sy.sector_configs(10, 5, 5, n, 32)
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), 3, 1)
    targets = pp.PreparedTargets(cfg_t, 3, distinct=True)
    if bits:
        _build_cores_with_narrow_hash(targets, bits, 90 + bits)
    occupied = np.nonzero(np.unpackbits(cfg, axis=1, bitorder="little"))[1].reshape(n, 10)
    for order in (2, 1):
        vals, starts, counts = _core_index(targets, order)
        per = 45 if order == 2 else 10
        assert counts.tolist()[:3] == [n * per, len(starts) - 1, 0]
        removed = [(a, b) for b in range(10) for a in range(b)] if order == 2 else [(a,) for a in range(10)]
        cores: dict[tuple[int, ...], set[int]] = {}
        for row, sites in enumerate(occupied.tolist()):
            for pick in removed:
                value = (row << 16) | (sites[pick[-1]] << 8 | sites[pick[0]] if order == 2 else sites[pick[0]])
                cores.setdefault(tuple(x for i, x in enumerate(sites) if i not in pick), set()).add(value)
        st = (starts & 0x7FFFFFFF).astype(np.int64)
        groups = [set(vals[a:b].tolist()) for a, b in zip(st[:-1], st[1:])]
        assert sum(len(g) for g in groups) == n * per
        where = {v: g for g, members in enumerate(groups) for v in members}
        held = [set() for _ in groups]  # the cores of each group
        for core, members in cores.items():
            (g,) = {where[v] for v in members}
            held[g].add(core)
        assert [len(h) > 1 for h in held] == (starts[:-1] >> 31).astype(bool).tolist()
    psi, g = sy.random_psi(n, 33), sy.random_psi(n, 34)
    want, asum, _ = orc.apply_within(1, cfg, psi, cfg, s, k, c)
    vec = torch.view_as_real(_dev(psi, cuda_device)).contiguous()
    got = pp.apply(terms, targets, cfg_t, vec, pp.MODE_FORWARD, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    assert np.all(np.abs(got[:, 0] + 1j * got[:, 1] - want) <= 1e-12 * asum + 1e-300)
    gvec = torch.view_as_real(_dev(g, cuda_device)).contiguous()
    ref, rsum, _ = orc.apply_within(1, cfg, g, cfg, s, k, c)  # the table is Hermitian
    got = pp.apply(terms, targets, cfg_t, gvec, pp.MODE_ADJOINT, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    assert np.all(np.abs(got[:, 0] + 1j * got[:, 1] - ref) <= 1e-12 * rsum + 1e-300)


@pytest.mark.parametrize("bits", [0, 4])
@pytest.mark.parametrize("order,size", [(2, 63), (2, 64), (2, 65), (2, 128), (2, 129), (2, 256), (1, 63), (1, 64), (1, 65), (1, 127)])
def test_groups_around_the_row_tiles(cuda_device: torch.device, order: int, size: int, bits: int) -> None:
    """Core groups on both sides of multiples of the 64 rows one wave takes, alone under their key and
    (4-bit hash columns) mixed with others: `size` site pairs of opposite parity beside each of 20
    spectators (order 2), or `size` sites beside one occupied site (order 1)."""
    if order == 2:
        nq = 9
        pairs = [(a, b) for a in range(0, 32, 2) for b in range(1, 32, 2)][:size]
        occupied = [(a, b, s) for a, b in pairs for s in range(40, 60)]
        table = _pair_heavy_table(np.arange(32), 6000, 7)
    else:
        nq = 16
        occupied = [(0, x) for x in range(1, size + 1)]
        table = _pair_heavy_table(np.arange(0, 128), 12000, 8)
    rows = np.zeros((len(occupied), 8 * nq), dtype=np.uint8)
    for row, sites in zip(rows, occupied):
        row[list(sites)] = 1
    cfg = sy.sort_unique_configs(np.packbits(rows, axis=1, bitorder="little"))
    n = len(cfg)
    s, k, c = table
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, 1)
    targets = pp.PreparedTargets(cfg_t, nq, distinct=True)
    if bits:
        _build_cores_with_narrow_hash(targets, bits, 50 + bits)
    _, starts, _ = _core_index(targets, order)
    st = (starts & 0x7FFFFFFF).astype(np.int64)
    assert np.diff(st).max() >= size
    psi = sy.random_psi(n, 33)
    vec = torch.view_as_real(_dev(psi, cuda_device)).contiguous()
    want, asum, _ = orc.apply_within(1, cfg, psi, cfg, s, k, c)
    got = pp.apply(terms, targets, cfg_t, vec, pp.MODE_FORWARD, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    assert np.all(np.abs(got[:, 0] + 1j * got[:, 1] - want) <= 1e-12 * asum + 1e-300)
    plain = pp.apply(terms, targets, cfg_t, vec, pp.MODE_ADJOINT, symmetric=pp.SYMMETRIC_OFF, pairs=False).cpu().numpy()
    got = pp.apply(terms, targets, cfg_t, vec, pp.MODE_ADJOINT, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    assert np.abs(got - plain).max() <= 1e-12 * (np.abs(c).sum() * np.abs(psi).max())


@pytest.mark.parametrize("size,shared,finite", [(80, True, True), (80, False, True), (129, True, True), (129, False, True), (80, True, False)])
def test_panels_of_large_groups(cuda_device: torch.device, size: int, shared: bool, finite: bool) -> None:
    """An index of over 2^25 entries takes its groups above 64 entries in panels of eight: groups of `size`
    site pairs beside two of 36 spectators, the same pairs in each or random ones (dense products over a
    small or a large union of slots), and the groups that the spectators make; with an infinite coefficient
    no panel is dense."""
    nq, rng = 16, np.random.default_rng(size)
    grid = [(a, b) for a in range(0, 32, 2) for b in range(1, 32, 2)]
    combos = [(s, t) for s in range(32, 68) for t in range(32, s)]
    combos = [combos[q] for q in rng.permutation(len(combos))[: 50_400 // size]]
    rows = np.zeros((len(combos) * size, 8 * nq), dtype=np.uint8)
    for k, (s, t) in enumerate(combos):
        picked = range(size) if shared else rng.permutation(len(grid))[:size]
        for j, q in enumerate(picked):
            rows[k * size + j, [*grid[q], s, t]] = 1
    rows[:, 68:] = 1
    cfg = sy.sort_unique_configs(np.packbits(rows, axis=1, bitorder="little"))
    n = len(cfg)
    assert n == len(rows) and n * (64 * 63 // 2) >= 1 << 25
    s, k, c = _pair_heavy_table(np.arange(48), 8000, 9)
    c[:, 1] = 0.0
    if not finite:
        s = np.concatenate([s, np.array([[60, 62, 120, 122]], dtype=np.int16)])  # its target pair is held by every row
        k = np.concatenate([k, np.array([[1, 1, 0, 0]], dtype=np.uint8)])
        c = np.concatenate([c, np.array([[np.inf, 0.0]])])
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, 1)
    targets = pp.PreparedTargets(cfg_t, nq, distinct=True)
    assert terms.pairs_desc.real == 1
    _, starts, _ = _core_index(targets, 2)
    sizes = np.diff((starts & 0x7FFFFFFF).astype(np.int64))[starts[:-1] >> 31 == 0]
    assert (sizes > 64).sum() >= 8 * 128  # panels enough
    psi, g = sy.random_psi(n, 33), sy.random_psi(n, 34)
    vec, gvec = (torch.view_as_real(_dev(x, cuda_device)).contiguous() for x in (psi, g))
    want, asum, _ = orc.apply_within(1, cfg, psi, cfg, s, k, c)
    got = pp.apply(terms, targets, cfg_t, vec, pp.MODE_FORWARD, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    assert np.all(np.abs(got[:, 0] + 1j * got[:, 1] - want) <= 1e-12 * asum + 1e-300)
    bound = 1e-12 * np.abs(c[np.isfinite(c[:, 0])]).sum()
    plain = pp.apply(terms, targets, cfg_t, gvec, pp.MODE_ADJOINT, symmetric=pp.SYMMETRIC_OFF, pairs=False).cpu().numpy()
    got = pp.apply(terms, targets, cfg_t, gvec, pp.MODE_ADJOINT, symmetric=pp.SYMMETRIC_OFF, pairs=True).cpu().numpy()
    assert np.abs(got - plain).max() <= bound * np.abs(g).max()


def _panel_kinds(targets: pp.PreparedTargets, most: int = 400) -> dict[str, int]:
    """What the panels of eight groups above 64 entries of the order-2 index are: dense (at least 20 pairs of
    entries per 16 x 16 x 4 product of the slots they use), sparse, or wide (over 960 slots); the largest
    group under "largest".  Up to `most` panels of a size range are looked at."""
    desc, buf = targets.cores(2), targets._cores[2][0]  # pylint: disable=protected-access

    def view(pointer: int, n: int, dtype: torch.dtype) -> np.ndarray:
        off = int(pointer) - buf.data_ptr()
        return buf[off:off + n * dtype.itemsize].view(dtype).cpu().numpy()

    bins = view(desc.bins, 3 * 39 + 40, torch.int32).astype(np.int64)
    groups, list_base = bins[:39], bins[78:117]
    glist = view(desc.glist, 2 * (int(list_base[38]) + int(groups[38])), torch.int32).astype(np.int64).reshape(-1, 2) & 0xFFFFFFFF
    slots = (view(desc.mvals, int(desc.capacity), torch.int64) >> 32) & 0xFFFF
    kinds = {"dense": 0, "sparse": 0, "wide": 0, "largest": 0, "panels": 0}
    for which, tiles in ((33, 2), (34, 2), (35, 3), (36, 4), (37, 5)):
        panels = -(-int(groups[which]) // (8 * tiles))
        kinds["panels"] += panels
        for k in range(min(panels, most)):
            lo = int(list_base[which]) + 8 * tiles * k
            items = glist[lo:min(lo + 8 * tiles, int(list_base[which] + groups[which]))]
            sizes = [(int(x), int(y) & 0xFFFF) for x, y in items if y >> 16 == 0]
            used = len(np.unique(np.concatenate([slots[x:x + n] for x, n in sizes]))) if sizes else 0
            pairs = sum(n * n for _, n in sizes)
            kinds["wide" if used > 960 else ("dense" if pairs >= 80 * (-(-used // 16)) ** 2 else "sparse")] += 1
            kinds["largest"] = max([kinds["largest"], *(n for _, n in sizes)])
    return kinds


def _hops_and_pairs(sites: int, n_terms: int, seed: int) -> tuple[np.ndarray, np.ndarray, np.ndarray]:
    """A real non-Hermitian table of pair excitations, hops and diagonal terms on the first `sites` sites."""
    rng = np.random.default_rng(seed)
    site = rng.permuted(np.tile(np.arange(sites), (n_terms, 1)), axis=1)[:, :4].astype(np.int16)
    kind = np.tile(np.array([1, 1, 0, 0], dtype=np.uint8), (n_terms, 1))
    u = rng.random(n_terms)
    kind[u < 0.2] = [1, 0, 2, 2]
    kind[u < 0.1] = [1, 0, 2, 2]
    site[u < 0.1, 1] = site[u < 0.1, 0]
    site[u < 0.2, 2:] = 0
    return site, kind, np.stack([rng.normal(size=n_terms), np.zeros(n_terms)], axis=1)


@pytest.mark.parametrize("case", ["one-word", "one-word-hard-core", "sparse", "wide", "above-256"])
def test_panels_with_two_vectors(cuda_device: torch.device, case: str) -> None:
    """The panels with one vector and with two, forward and adjoint, where they are dense products and where
    they are walked (too few pairs for the slots they use, or more slots than the LDS holds): one-word
    configs, fermions and hard-core bosons, groups up to and above 256 entries."""
    pc = 2 if case.endswith("hard-core") else 1
    if case.startswith("one-word"):
        s, k, c = sorted_terms(*sy.molecular_terms(26, 5))
        c = c * np.where(np.random.default_rng(6).random(len(c)) < 0.5, 1.0, 0.5)[:, None]  # not Hermitian
        cfg, nq = sy.excitation_configs(26, 7, 7, 400_000, 7), 7
    else:
        # `size` random pairs of opposite parity on the first `of` sites beside every two of the next `spectators`, `fixed` more occupied
        of, size, spectators, fixed = {"sparse": (60, 90, 36, 32), "wide": (80, 400, 30, 18), "above-256": (36, 300, 50, 12)}[case]
        rng, nq = np.random.default_rng(size), 16
        grid = np.array([(a, b) for a in range(0, of, 2) for b in range(1, of, 2)])
        combos = [(of + x, of + y) for y in range(spectators) for x in range(y)]
        rows = np.zeros((len(combos) * size, 8 * nq), dtype=np.uint8)
        for j, (x, y) in enumerate(combos):
            part = rows[j * size:(j + 1) * size]
            part[:, [x, y]] = 1
            picked = grid[rng.permutation(len(grid))[:size]]
            part[np.arange(size), picked[:, 0]] = 1
            part[np.arange(size), picked[:, 1]] = 1
        rows[:, of + spectators:of + spectators + fixed] = 1
        cfg = sy.sort_unique_configs(np.packbits(rows, axis=1, bitorder="little"))
        s, k, c = _hops_and_pairs(of + spectators, 8000, 9)
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), nq, pc)
    targets = pp.PreparedTargets(cfg_t, nq, distinct=True)
    assert terms.pairs_desc.real == 1 and not terms.hermitian and terms.n_residual_terms == 0
    assert targets.cores(2).capacity >= 1 << 25
    kinds = _panel_kinds(targets)
    assert kinds["panels"] >= 128
    assert kinds[{"sparse": "sparse", "wide": "wide"}.get(case, "dense")] >= 8, kinds
    if case in ("wide", "above-256"):
        assert kinds["largest"] > 256
    vecs = [torch.view_as_real(_dev(sy.random_psi(len(cfg), seed), cuda_device)).contiguous() for seed in (33, 34)]
    for mode in (pp.MODE_FORWARD, pp.MODE_ADJOINT):
        plain = [pp.apply(terms, targets, cfg_t, v, mode, symmetric=pp.SYMMETRIC_OFF, pairs=False) for v in vecs]
        one = pp.apply(terms, targets, cfg_t, vecs[0], mode, symmetric=pp.SYMMETRIC_OFF, pairs=True)
        both = pp.apply_dual(terms, targets, *vecs, mode)
        for got, want, v in ((one, plain[0], vecs[0]), (both[0], plain[0], vecs[0]), (both[1], plain[1], vecs[1])):
            # rows meet at most a few thousand of the terms: the rounding of their sums against the largest products
            assert (got - want).abs().max().item() <= 1e-12 * np.abs(c).sum() * v.abs().max().item()


@pytest.mark.parametrize("bits", [0, 4])
@pytest.mark.parametrize("n_orb,electrons,n", [(4, 2, 36), (6, 2, 85), (10, 5, 11)])
def test_small_indexes_repeat_to_the_last_bit(cuda_device: torch.device, n_orb: int, electrons: int, n: int, bits: int) -> None:
    """An index of up to 512 entries (36 rows of 4 electrons: 216; 85: 510; 11 of 10: 495) is walked by one
    wave in a fixed order: fresh indexes and repeated applications agree to the last bit, in both modes,
    with the set's hash and with 4-bit hash columns (groups of many cores)."""
    s, k, c = sorted_terms(*sy.molecular_terms(n_orb, 41))
    cfg = sy.sector_configs(n_orb, electrons, electrons, n, 42)
    cfg_t = _dev(cfg, cuda_device)
    terms = pp.PreparedTerms(_dev(s, cuda_device), _dev(k, cuda_device), _dev(c, cuda_device), cfg.shape[1], 1)
    vec = torch.view_as_real(_dev(sy.random_psi(n, 43), cuda_device)).contiguous()
    first = {}
    for _ in range(8):
        targets = pp.PreparedTargets(cfg_t, cfg.shape[1], distinct=True)
        if bits:
            _build_cores_with_narrow_hash(targets, bits, 44)
        assert targets.cores(2).capacity <= 512
        for _again in range(3):
            for mode in (pp.MODE_FORWARD, pp.MODE_ADJOINT):
                got = pp.apply(terms, targets, cfg_t, vec, mode, symmetric=pp.SYMMETRIC_OFF, pairs=True).view(torch.int64)
                assert torch.equal(got, first.setdefault(mode, got))
