"""GPU parity of the lossy DAG (LSVDAG) row and its learned proposer.

* exhaustive proposer: every level array, every per-level statistic and the
  encoded .svdag of the lossy DAG are bit-exact against the oracle;
* learned proposer: given the kNN lists the GPU used (recorded), the oracle
  reproduces the whole lossy DAG bit-exactly; the kNN itself is bit-exact
  against the oracle's sequential restatement on the same embeddings;
* MLP forward / gradients against the NumPy oracle (bf16 rounding at the
  same points), with the tolerances written below: the GPU accumulates in a
  different order (MFMA), so an intermediate bf16 rounding can land one ulp
  (2^-8 relative) apart.
"""
import numpy as np
import pytest
import torch

import mlp_oracle as M
import oracle as O
from decode import decode_words

import svdag_amd as S
import svdag_amd.workloads as W
from test_oracle import clustered_codes, random_codes

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

SCENES = {
    "terrain7": lambda: (W.terrain_codes(7, seed=1), 7),
    "caves7": lambda: (W.cave_codes(7, seed=3), 7),
    "random6": lambda: (random_codes(6, 20000, 3), 6),
    "clustered7": lambda: (clustered_codes(7, 2), 7),
}

STAT_FIELDS = ("level", "bound", "nodes_before", "nodes_after", "candidates", "listed", "verified", "merged",
               "error_bound")


def gpu_dag(ctx, codes, L):
    g = S.Octree.from_morton(ctx, codes, L)
    g.to_dag()
    return g


def oracle_dag(codes, L):
    o = O.OracleOctree.from_morton(codes, L)
    o.to_dag()
    return o


def assert_same_dag(g, o, L):
    for l in range(L):
        np.testing.assert_array_equal(g.level(S.VIEW_DAG, l), o.level(l), err_msg=f"level {l}")
    assert g.counts()[0] == o.n_nodes


def assert_same_stats(st_g, st_o):
    for f in STAT_FIELDS:
        np.testing.assert_array_equal(st_g[f], st_o[f], err_msg=f)


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("mode", ["max10", "factor1", "refs3"])
def test_lossy_exhaustive_bit_exact(ctx, name, mode):
    codes, L = SCENES[name]()
    kw = {"max10": dict(max_diff=10), "factor1": dict(max_diff=0, diff_factor=1.0),
          "refs3": dict(max_diff=6, max_refs=3, list_cap=5)}[mode]
    print(f"[case] {name} {mode} L={L} voxels={codes.size}", flush=True)
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    st_g = g.lossy_merge(1, L - 2, **kw)
    st_o = o.lossy_merge(1, L - 2, **kw)
    assert_same_stats(st_g, st_o)
    assert_same_dag(g, o, L)
    assert st_g["merged"].sum() > 0 or mode == "refs3"
    g.encode(S.FMT_SVDAG)
    o.init_child_levels()
    assert g.encoded_bytes(S.FMT_SVDAG) == o.encode(0)
    # the lossy DAG feeds the symmetry pass and the SSVDAG encoder as usual
    g.to_sdag()
    g.encode(S.FMT_SSVDAG)
    o.to_sdag()
    assert g.encoded_bytes(S.FMT_SSVDAG) == o.encode(2)


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("mode", ["max10cap8", "factor1cap32", "refs3cap40"])
def test_lossy_ranked_bit_exact(ctx, name, mode):
    """The ranked exhaustive proposer (the list_cap nearest earlier nodes by
    Hamming distance, nearest first) equals the oracle's, level by level and
    statistic by statistic; the three list capacities take the 16-, 32- and
    64-entry register lists."""
    codes, L = SCENES[name]()
    kw = {"max10cap8": dict(max_diff=10, list_cap=8), "factor1cap32": dict(max_diff=0, diff_factor=1.0, list_cap=32),
          "refs3cap40": dict(max_diff=6, max_refs=3, list_cap=40)}[mode]
    print(f"[case] ranked {name} {mode} L={L} voxels={codes.size}", flush=True)
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    st_g = g.lossy_merge(1, L - 2, ranked=True, **kw)
    st_o = o.lossy_merge(1, L - 2, ranked=True, **kw)
    assert_same_stats(st_g, st_o)
    assert_same_dag(g, o, L)
    g.encode(S.FMT_SVDAG)
    o.init_child_levels()
    assert g.encoded_bytes(S.FMT_SVDAG) == o.encode(0)


@pytest.mark.parametrize("cap", [1, 2, 64])
@pytest.mark.parametrize("bound", [1, 24, 600])
def test_lossy_exhaustive_list_edges(ctx, cap, bound):
    """The matrix-core scan at its edges: lists that overflow twice their
    capacity (capacities 1, 2 and 64), bounds whose popcount window is one
    side of the range or all of it (600: every pair matches), levels of a few
    to a few thousand nodes (partial 32-row tiles and stages, one and several
    chunks)."""
    codes, L = random_codes(6, 20000, 3), 6
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    st_g = g.lossy_merge(1, L - 2, max_diff=bound, list_cap=cap)
    st_o = o.lossy_merge(1, L - 2, max_diff=bound, list_cap=cap)
    assert_same_stats(st_g, st_o)
    assert_same_dag(g, o, L)


@pytest.mark.parametrize("L", [4, 7, 8, 9, 10])
def test_lossy_exact_difference_depths(ctx, L):
    """Octants that are copies of one another but for a few voxels, so that
    nodes of every level are compared down to the occupancies three levels
    above the bottom: each nesting depth of the difference (level 1 of 4 to 8
    levels) and the stack walk beyond (9 and 10 levels)."""
    rng = np.random.default_rng(L)
    sub = 3 * (L - 1)
    base = np.unique(rng.integers(0, 1 << sub, 2500, dtype=np.uint64))
    parts = []
    for o in range(6):
        keep = np.ones(base.size, bool)
        keep[rng.choice(base.size, 2 * o, replace=False)] = False
        parts.append(base[keep] | np.uint64(o << sub))
    codes = np.unique(np.concatenate(parts))
    for bound in (3, 9):
        g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
        st_g = g.lossy_merge(1, L - 2, max_diff=bound)
        st_o = o.lossy_merge(1, L - 2, max_diff=bound)
        assert_same_stats(st_g, st_o)
        assert_same_dag(g, o, L)


def test_lossy_exhaustive_lists_of_a_large_level(ctx):
    """A level of some 260K nodes takes the two-tile workgroups.  At bound 1 no
    list fills, so the ranked proposer (its own kernel, every earlier node)
    lists the same pairs: the listed and verified counts agree."""
    codes, L = random_codes(9, 1500000, 5), 9
    st = []
    for ranked in (False, True):
        g = gpu_dag(ctx, codes, L)
        assert g.level_size(S.VIEW_DAG, 6) > 200000
        st.append(g.lossy_merge(6, 6, max_diff=1, list_cap=64, ranked=ranked))
        g.free()
    assert st[0]["listed"][0] > 0
    for f in ("candidates", "listed", "verified"):
        np.testing.assert_array_equal(st[0][f], st[1][f], err_msg=f)


@pytest.mark.parametrize("two_tiles,voxels,bound,cap", [(False, 380000, 4, 16), (True, 800000, 6, 1),
                                                         (True, 800000, 8, 2), (True, 800000, 8, 64),
                                                         (True, 800000, 24, 16)])
def test_lossy_exhaustive_full_lists_of_a_large_level(ctx, two_tiles, voxels, bound, cap):
    """Lists of a large level that overflow twice their capacity, and nodes
    that stop between chunks (bounds that fill a list within a few thousand
    nodes, and bounds that leave some open to the end), by both workgroup
    shapes: the merged level equals the oracle's, which walks the earlier nodes
    in order."""
    codes, L = random_codes(9, voxels, 5), 9
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert (g.level_size(S.VIEW_DAG, 6) >= 768 * cus) == two_tiles
    kw = dict(max_diff=bound, list_cap=cap)
    st_g, st_o = g.lossy_merge(6, 6, **kw), o.lossy_merge(6, 6, **kw)
    assert_same_stats(st_g, st_o)
    assert_same_dag(g, o, L)


def test_lossy_error_within_accounted_bound(ctx):
    codes, L = W.cave_codes(7, seed=3), 7
    g = gpu_dag(ctx, codes, L)
    st = g.lossy_merge(1, L - 2, max_diff=10)
    g.encode(S.FMT_SVDAG)
    vox = decode_words(g.encoded_bytes(S.FMT_SVDAG), False)
    diff = np.setxor1d(vox, codes).size
    assert 0 < diff <= int(st["error_bound"].sum()), (diff, st["error_bound"])


def test_lossy_signatures_match_oracle(ctx):
    codes, L = W.terrain_codes(7, seed=1), 7
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    for lev in range(1, L - 1):
        n = g.level_size(S.VIEW_DAG, lev)
        sig = torch.zeros(n * 16, dtype=torch.int32, device=DEV)
        torch.cuda.synchronize()
        g.lossy_signatures(lev, sig.data_ptr())
        np.testing.assert_array_equal(sig.cpu().numpy().view(np.uint32).reshape(n, 16), o.lossy_signatures(lev))


@pytest.mark.parametrize("L", [3, 4, 6])
def test_lossy_signatures_every_level(ctx, L):
    """The root and the two levels above the voxels, whose occupancies end
    before 512 bits."""
    codes = random_codes(L, 40 * L, seed=L)
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    for lev in range(L):
        n = g.level_size(S.VIEW_DAG, lev)
        sig = torch.full((n * 16,), -1, dtype=torch.int32, device=DEV)
        torch.cuda.synchronize()
        g.lossy_signatures(lev, sig.data_ptr())
        ctx.sync()
        np.testing.assert_array_equal(sig.cpu().numpy().view(np.uint32).reshape(n, 16), o.lossy_signatures(lev))


def test_signatures_do_not_wait_for_other_streams(ctx):
    """The caller orders its own work: a call runs beside what is pending on
    the default stream (a spinning kernel of some milliseconds)."""
    codes, L = W.terrain_codes(7, seed=1), 7
    g = gpu_dag(ctx, codes, L)
    sig = torch.zeros(g.level_size(S.VIEW_DAG, 4) * 16, dtype=torch.int32, device=DEV)
    g.lossy_signatures(4, sig.data_ptr())
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    torch.cuda._sleep(20_000_000)
    done.record()
    g.lossy_signatures(4, sig.data_ptr())
    assert not done.query()
    torch.cuda.synchronize()


def test_lossy_argument_errors(ctx):
    codes, L = W.terrain_codes(6, seed=1), 6
    g = gpu_dag(ctx, codes, L)
    for bad in (dict(lev_lo=0, lev_hi=3), dict(lev_lo=2, lev_hi=5), dict(lev_lo=3, lev_hi=2)):
        with pytest.raises(S.SvdError):
            g.lossy_merge(bad["lev_lo"], bad["lev_hi"], max_diff=4)
    with pytest.raises(S.SvdError):
        g.lossy_merge(1, 4, max_diff=4, list_cap=65)
    sv = S.Octree.from_morton(ctx, codes, L)          # still an SVO
    with pytest.raises(S.SvdError):
        sv.lossy_merge(1, 4, max_diff=4)


# ---------------------------------------------------------------- MLP
def _rand_sigs(n, seed, density=0.15):
    rng = np.random.default_rng(seed)
    bits = (rng.random((n, 16, 32)) < density).astype(np.uint64)
    return (bits << np.arange(32, dtype=np.uint64)).sum(axis=2).astype(np.uint32)


def _dev_u32(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).to(DEV)


def test_mlp_init_matches_oracle(ctx):
    m = S.MLP(ctx, seed=5)
    np.testing.assert_array_equal(m.params(), M.init_params(5))


def test_mlp_forward_matches_oracle(ctx):
    m = S.MLP(ctx, seed=3)
    p = M.init_params(3)
    p[M.split(p)[0].size:M.split(p)[0].size + 256] = np.linspace(-0.1, 0.1, 256, dtype=np.float32)   # b1
    m.set_params(p)
    n = 1000
    sig = _rand_sigs(n, 1)
    emb = torch.zeros(n * 32, dtype=torch.float32, device=DEV)
    dsig = _dev_u32(sig)                 # keep the tensor alive while the library reads it
    torch.cuda.synchronize()
    m.embed(dsig.data_ptr(), n, emb.data_ptr())
    e_g = emb.cpu().numpy().reshape(n, 32)
    e_o, _ = M.forward(p, M.unpack_bits(sig))
    scale = np.abs(e_o).max()
    # one bf16 ulp (2^-8) of a hidden activation moves e by far less than 1% of its range
    assert np.abs(e_g - e_o).max() <= 1e-2 * scale, np.abs(e_g - e_o).max() / scale
    assert np.corrcoef(e_g.ravel(), e_o.ravel())[0, 1] > 0.9999


@pytest.mark.parametrize("P", [16, 48, 256, 4112])
def test_mlp_gradients_match_oracle(ctx, P):
    """Batches of one workgroup, a partial split of the weight gradients, several
    splits, and more workgroups than compute units."""
    m = S.MLP(ctx, seed=9)
    p = M.init_params(9)
    sig = _rand_sigs(2 * P, 2)
    sig[1::2] = sig[0::2] ^ (_rand_sigs(P, 3, density=0.02))     # near pairs
    H = M.hamming(sig[0::2], sig[1::2])
    # both tensors stay referenced: a freed temporary's block is reused by the next allocation
    dsig, dlab = _dev_u32(sig), _dev_u32(H.astype(np.uint32))
    torch.cuda.synchronize()
    loss_g, grad_g = m.loss_grad(dsig.data_ptr(), dlab.data_ptr(), P)
    loss_o, grad_o = M.loss_and_grads(p, M.unpack_bits(sig), H)
    errs = {"loss": abs(loss_g - loss_o) / abs(loss_o)}
    off = 0
    for name, t in zip(("W1", "b1", "W2", "b2", "W3", "b3"), M.split(p)):
        a, b = grad_g[off:off + t.size], grad_o[off:off + t.size]
        off += t.size
        errs[name] = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
    print({k: f"{v:.2e}" for k, v in errs.items()}, flush=True)
    # the GPU accumulates in MFMA order: an activation or delta whose bf16
    # rounding lands one ulp (2^-8) apart moves the loss by ~1e-5 and the
    # gradients by ~1e-2 relative (near pairs cancel in e_a - e_b)
    assert errs["loss"] <= 1e-3
    for name in ("W1", "b1", "W2", "b2", "W3", "b3"):
        assert errs[name] <= 3e-2, (name, errs[name])


def test_mlp_training_reduces_loss(ctx):
    codes, L = W.cave_codes(7, seed=3), 7
    g = gpu_dag(ctx, codes, L)
    m = S.MLP(ctx, seed=1)
    st = m.train(g, 2, L - 2, pairs_per_step=512, steps=300, lr=2e-3, seed=5)
    print(f"loss {st.first_loss:.3f} -> {st.last_loss:.3f} over {st.pairs} pairs, {st.ms_train:.1f} ms", flush=True)
    assert st.last_loss < 0.5 * st.first_loss


# ---------------------------------------------------------------- kNN
def test_knn_matches_oracle(ctx):
    rng = np.random.default_rng(4)
    n = 3000
    e = (rng.standard_normal((n, 32)) * np.linspace(2, 0.1, 32)).astype(np.float32)
    e[100] = e[7]                       # an exact duplicate (distance 0, tie by index)
    de = torch.from_numpy(e).to(DEV)
    out = torch.zeros(n * 16, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    ctx.knn(de.data_ptr(), n, 16, 4, 16, 32, 7, out.data_ptr())
    got = out.cpu().numpy().view(np.uint32).reshape(n, 16)
    np.testing.assert_array_equal(got, O.knn_lsh(e, 16, 4, 16, 32, 7))
    assert got[7, 0] == 100 and got[100, 0] == 7
    # signature re-ranking
    sig = _rand_sigs(n, 6, density=0.1)
    dsig = _dev_u32(sig)
    torch.cuda.synchronize()
    ctx.knn(de.data_ptr(), n, 16, 4, 12, 48, 9, out.data_ptr(), sig_ptr=dsig.data_ptr())
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32).reshape(n, 16),
                                  O.knn_lsh(e, 16, 4, 12, 48, 9, sig=sig))


@pytest.mark.parametrize("n,k,tables,bits,window", [(1, 16, 2, 4, 64), (31, 16, 2, 4, 3), (33, 1, 3, 4, 1),
                                                    (128, 16, 2, 3, 96), (129, 7, 2, 3, 95), (300, 16, 9, 5, 63),
                                                    (1000, 15, 3, 24, 96), (1000, 17, 2, 6, 40)])
def test_knn_signature_windows(ctx, n, k, tables, bits, window):
    """The matrix-core windows at their edges: fewer points than a workgroup,
    one or a partial query tile, windows of 1 to 96 positions (partial row
    tiles), several tables over the same neighbours (candidates the list
    already holds), many equal distances and equal signatures, and k = 17
    (the general kernel)."""
    rng = np.random.default_rng(n + k)
    sig = _rand_sigs(max(n // 3, 1), 11 + n, density=0.02)[rng.integers(0, max(n // 3, 1), n)]
    e = rng.standard_normal((n, 32)).astype(np.float32)
    de, dsig = torch.from_numpy(e).to(DEV), _dev_u32(sig)
    out = torch.zeros(n * k, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    ctx.knn(de.data_ptr(), n, k, tables, bits, window, 9, out.data_ptr(), sig_ptr=dsig.data_ptr())
    ctx.sync()
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32).reshape(n, k),
                                  O.knn_lsh(e, k, tables, bits, window, 9, sig=sig))


def test_knn_full_window_is_brute_force(ctx):
    rng = np.random.default_rng(5)
    n = 90                               # every point within +-96 positions of every other
    e = rng.standard_normal((n, 32)).astype(np.float32)
    de = torch.from_numpy(e).to(DEV)
    out = torch.zeros(n * 8, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    ctx.knn(de.data_ptr(), n, 8, 1, 4, 96, 3, out.data_ptr())
    got = out.cpu().numpy().view(np.uint32).reshape(n, 8)
    d = np.zeros((n, n), np.float32)           # the same sequential fp32 sum as the kernel
    for k in range(32):
        t = e[:, None, k] - e[None, :, k]
        d = d + t * t
    np.fill_diagonal(d, np.inf)
    want = np.argsort(d, axis=1, kind="stable")[:, :8]
    np.testing.assert_array_equal(got, want)


def test_knn_of_more_points_than_22_bits(ctx):
    """Beyond 2^22 points a (distance, node) key no longer fits 32 bits: the
    window kernel that keeps them apart, at its list size of 16, over two
    tables and many equal signatures."""
    n = (1 << 22) + 777
    rng = np.random.default_rng(3)
    e = rng.standard_normal((n, 32), dtype=np.float32)
    sig = (rng.integers(0, 1 << 32, (n // 4, 16), dtype=np.uint32) &
           rng.integers(0, 1 << 32, (n // 4, 16), dtype=np.uint32))[rng.integers(0, n // 4, n)]
    de, dsig = torch.from_numpy(e).to(DEV), _dev_u32(sig)
    out = torch.zeros(n * 16, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    ctx.knn(de.data_ptr(), n, 16, 2, 12, 3, 9, out.data_ptr(), sig_ptr=dsig.data_ptr())
    ctx.sync()
    print(f"[case] {n} points searched", flush=True)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32).reshape(n, 16),
                                  O.knn_lsh(e, 16, 2, 12, 3, 9, sig=sig))


# ---------------------------------------------------------------- learned lossy
def test_knn_refine_of_more_nodes_than_22_bits(ctx):
    """A level of more than 2^22 nodes takes the refinement with 64-bit keys."""
    L, lev, k = 11, 8, 2
    gen = torch.Generator(device=DEV).manual_seed(7)
    codes = torch.unique(torch.randint(0, 1 << (3 * L), (36_000_000,), dtype=torch.int64, device=DEV, generator=gen))
    torch.cuda.synchronize()
    g, m = S.Octree.from_morton(ctx, (codes.data_ptr(), codes.numel()), L), S.MLP(ctx, seed=1)
    g.to_dag()
    n = g.level_size(S.VIEW_DAG, lev)
    print(f"[case] {codes.numel()} voxels, {n} nodes in level {lev}", flush=True)
    assert n > 1 << 22
    dsig = torch.zeros(n * 16, dtype=torch.int32, device=DEV)
    demb = torch.zeros(n * 32, dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    g.lossy_signatures(lev, dsig.data_ptr())
    m.embed(dsig.data_ptr(), n, demb.data_ptr())
    ctx.sync()
    sig, emb = dsig.cpu().numpy().view(np.uint32).reshape(n, 16), demb.cpu().numpy().reshape(n, 32)
    kw = dict(k=k, tables=1, bits=12, window=2)
    _, rec = g.lossy_merge(lev, lev, max_diff=1, model=m, refine=1, record_knn=True, **kw)
    g.free()
    print("[case] merged", flush=True)
    want = O.knn_refine(sig, O.knn_lsh(emb, k, 1, 12, 2, 7, sig=sig), 1)
    np.testing.assert_array_equal(rec[:n * k].reshape(n, k), want)


@pytest.mark.parametrize("k,rounds", [(1, 1), (15, 2), (16, 1), (16, 3), (17, 2), (32, 1)])
def test_knn_refine_list_sizes(ctx, k, rounds):
    """Refinement with 32-bit keys (k <= 16) and 64-bit ones, after an odd and
    an even number of rounds: the recorded lists equal the oracle's."""
    codes, L = W.cave_codes(6, seed=4), 6
    g, m = gpu_dag(ctx, codes, L), S.MLP(ctx, seed=1)
    n = g.level_size(S.VIEW_DAG, L - 2)
    dsig = torch.zeros(n * 16, dtype=torch.int32, device=DEV)
    demb = torch.zeros(n * 32, dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    g.lossy_signatures(L - 2, dsig.data_ptr())
    m.embed(dsig.data_ptr(), n, demb.data_ptr())
    ctx.sync()
    sig, emb = dsig.cpu().numpy().view(np.uint32).reshape(n, 16), demb.cpu().numpy().reshape(n, 32)
    _, rec = g.lossy_merge(L - 2, L - 2, max_diff=10, model=m, k=k, refine=rounds, record_knn=True)
    want = O.knn_refine(sig, O.knn_lsh(emb, k, 8, 16, 64, 7, sig=sig), rounds)
    np.testing.assert_array_equal(rec[:n * k].reshape(n, k), want)


def test_lossy_learned_matches_oracle_given_knn(ctx):
    codes, L = W.cave_codes(7, seed=3), 7
    g, o = gpu_dag(ctx, codes, L), oracle_dag(codes, L)
    m = S.MLP(ctx, seed=1)
    m.train(g, 1, L - 2, pairs_per_step=512, steps=200, lr=2e-3, seed=5)
    # the first processed level (L-2) sees the input DAG: its kNN lists are
    # checked against the oracle's search on the same signatures / embeddings
    n0 = g.level_size(S.VIEW_DAG, L - 2)
    dsig = torch.zeros(n0 * 16, dtype=torch.int32, device=DEV)
    demb = torch.zeros(n0 * 32, dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    g.lossy_signatures(L - 2, dsig.data_ptr())
    m.embed(dsig.data_ptr(), n0, demb.data_ptr())
    sig0 = dsig.cpu().numpy().view(np.uint32).reshape(n0, 16)
    emb0 = demb.cpu().numpy().reshape(n0, 32)
    st_g, rec = g.lossy_merge(1, L - 2, max_diff=10, model=m, record_knn=True)
    lsh = O.knn_lsh(emb0, 16, 8, 16, 64, 7, sig=sig0)
    np.testing.assert_array_equal(rec[:n0 * 16].reshape(n0, 16), O.knn_refine(sig0, lsh, 2))
    st_o = o.lossy_merge(1, L - 2, max_diff=10, proposals=rec, k=16, list_cap=32)
    assert_same_stats(st_g, st_o)
    assert_same_dag(g, o, L)
    assert st_g["merged"].sum() > 0


def test_learned_proposer_gains_over_untrained(ctx):
    """What the trained encoder adds: with the neighbour search alone (no
    neighbour-of-neighbour rounds) the trained embedding finds more merges
    than the untrained one, and the refinement rounds close most of the rest
    of the gap to the exhaustive proposer.  (At 256^3 the full pipeline ends
    about 4% above exhaustive; on the 4096^3 cave measurement it ends 0.5%
    below it.)"""
    codes, L = W.cave_codes(8, seed=3), 8
    res = {}
    g = gpu_dag(ctx, codes, L)
    st = g.lossy_merge(2, L - 2, max_diff=10)
    res["exhaustive"] = (g.counts()[0], int(st["merged"].sum()))
    trained = S.MLP(ctx, seed=1)
    trained.train(gpu_dag(ctx, codes, L), 2, L - 2, pairs_per_step=1024, steps=400, lr=2e-3, seed=5, near_pct=80)
    untrained = S.MLP(ctx, seed=1)
    for tag, m, refine in (("untrained-r0", untrained, 0), ("trained-r0", trained, 0), ("trained-r2", trained, 2)):
        g = gpu_dag(ctx, codes, L)
        st = g.lossy_merge(2, L - 2, max_diff=10, model=m, refine=refine)
        res[tag] = (g.counts()[0], int(st["merged"].sum()))
    print(res, flush=True)
    assert res["trained-r0"][0] < res["untrained-r0"][0]
    assert res["trained-r0"][1] > res["untrained-r0"][1]
    assert res["trained-r2"][0] < res["trained-r0"][0]
    assert res["trained-r2"][0] <= 1.05 * res["exhaustive"][0]
