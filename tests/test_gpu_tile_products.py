"""Products in tiles with their ends (csrc/gemm_tile.hip), and which of them a shape runs with, against 64 bits."""
import json

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(m, n, k, gated, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * n if gated else n, k, device=DEV, generator=g) / k ** 0.5).to(torch.bfloat16)
    return a, w


def _want(a, w, n, end, start=None):
    z = a.double() @ w.double().T
    if end == "gated":
        return torch.nn.functional.silu(z[:, :n]) * z[:, n:]
    if end == "add":
        return start.double() + z
    return {None: lambda x: x, "silu": torch.nn.functional.silu, "relu2": lambda x: torch.relu(x) ** 2,
            "gelu": torch.nn.functional.gelu}[end](z)


def _close(got, want, name):
    # one rounding to bfloat16 (2^-9 of the value) and sums of products of unit spread in float: far below 1e-4
    err = (got.double() - want).abs()
    assert bool((err <= 2.0 ** -8 * want.abs() + 1e-4).all()), f"{name}: {float(err.max())}"


SHAPES = 13


def test_every_shape_is_tested():
    from dinfer_amd.kernels import tiles
    assert len(tiles.shapes()) == SHAPES


@pytest.mark.parametrize("shape", range(SHAPES))
def test_every_shape_at_its_edges(shape):
    """Rows and columns one below, at and one above a tile, the least depth, one more step, and more tiles than workgroups (several
    rounds of a walk); nothing outside of the product is written."""
    from dinfer_amd.kernels import ops, tiles
    rows, cols, least, gated_ok = tiles.shapes()[shape]
    sizes = [(1, 8, least), (rows - 1, cols - 8, least), (rows, cols, least + 64), (rows + 1, cols + 8, least),
             (3 * rows + 17, 2 * cols + 40, least + 192), (19 * rows - 5, 17 * cols + 24, least)]
    for m, n, k in sizes:
        for end in (None, "add", "relu2", "silu", "gelu") + (("gated",) if gated_ok else ()):
            if end in ("silu", "gelu") and m > 4 * rows:
                continue
            a, w = _inputs(m + 5, n, k, end == "gated", seed=m)
            buf = torch.full((m + 9, n + 8), 3.0, device=DEV, dtype=torch.bfloat16)
            out = buf[2:m + 7, :n]
            start = out.clone()
            ops.gemm_tile(a, w, out, m, shape, add=end == "add", gated=end == "gated", act=end if end in ops.GEMM_TILE_ACTS else None)
            _close(out[:m], _want(a[:m], w, n, end, start[:m]), f"{m}x{n}x{k} {end}")
            assert bool((buf[:2] == 3).all()) and bool((buf[m + 2:] == 3).all()) and bool((buf[:, n:] == 3).all())
        a, w = _inputs(m + 5, n, k, False, seed=m)
        buf = torch.full((m + 9, n + 8), 3.0, device=DEV)
        ops.gemm_tile(a, w, buf[2:m + 7, :n], m, shape)
        # sums of k products of size k^-1/2 in float: at most k^1/2 2^-24 off, with room for their order
        torch.testing.assert_close(buf[2:m + 2, :n].double(), _want(a[:m], w, n, None), rtol=0, atol=4 * k ** 0.5 * 2.0 ** -24 * 8)
        assert bool((buf[:2] == 3).all()) and bool((buf[m + 2:] == 3).all()) and bool((buf[:, n:] == 3).all())


def test_what_the_tiles_refuse():
    from dinfer_amd.kernels import lib, ops
    a, w = _inputs(64, 64, 512, False)
    out = torch.zeros(64, 64, device=DEV, dtype=torch.bfloat16)
    for bad in (lambda: ops.gemm_tile(a[:, :500], w[:, :500], out, 64, 0),                      # depth
                lambda: ops.gemm_tile(a, w[:60], out[:, :60], 64, 0),                           # columns
                lambda: ops.gemm_tile(a[:, 4:452], w[:, :448], out, 64, 0),                     # alignment
                lambda: ops.gemm_tile(a[:, :64], w[:, :64], out, 64, 0),                        # fewer steps than it keeps ahead
                lambda: ops.gemm_tile(a, w, out, 64, 99)):                                      # no such shape
        with pytest.raises(lib.KernelError):
            bad()
    assert bool((out == 0).all())


def test_products_with_ends_choose_and_remember(tmp_path):
    """Nothing is chosen outside measuring(); inside, a choice is made and kept in the plan file, from which another process takes it;
    whichever runs, the result is the same to its rounding. Operands off 16 bytes take the separate pass."""
    from dinfer_amd.kernels import blaslt, gemm
    blaslt.configure(tuning="measured", plan_file=str(tmp_path / "plans.json"))
    blaslt._plans.clear()
    blaslt._ends.clear()
    cases = [(200, 384, 512), (1040, 512, 1024), (300, 200, 500), (96, 72, 64)]

    def run():
        for m, n, k in cases:
            for end in ("gated", "relu2", "gelu_tanh"):
                a, w = _inputs(m + 40, n, k, end == "gated")
                out = torch.zeros(m + 40, n, device=DEV, dtype=torch.bfloat16)
                scratch = torch.empty(m + 40, 2 * n, device=DEV, dtype=torch.bfloat16)
                if end == "gated":
                    gemm.gated_nt(a, w, out, scratch, m, "silu")
                else:
                    gemm.act_nt(a, w, out, m, end)
                z = a[:m].double() @ w.double().T
                want = (_want(a[:m], w, n, end) if end != "gelu_tanh" else torch.nn.functional.gelu(z, approximate="tanh"))
                # a pass of its own rounds the product first: 2^-9 of each factor, and the activations' slopes are at most 2 |z| + 1.2
                err = (out[:m].double() - want).abs()
                bound = 2.0 ** -7 * want.abs() + 2.0 ** -8 * (z.abs().amax(-1, keepdim=True) * 2 + 1.2)
                assert bool((err <= bound).all()), f"{m}x{n}x{k} {end}"

    try:
        run()
        assert not any(p.tuned and p.tile for p in blaslt._ends.values())
        with blaslt.measuring():
            run()
        stored = json.loads((tmp_path / "plans.json").read_text())
        assert any(k.endswith(",gated") for k in stored) and any(k.endswith(",relu2") for k in stored)
        chosen = {k: p.tile and p.tile.shape for k, p in blaslt._ends.items() if p.tuned}
        assert any(p.times for p in blaslt._ends.values())
        blaslt._plans.clear()
        blaslt._ends.clear()
        run()
        assert {k: p.tile and p.tile.shape for k, p in blaslt._ends.items() if p.tuned} == chosen
        assert all(p.times is None for p in blaslt._ends.values())
        # one column further: rows on 16 bytes no longer
        a, w = _inputs(240, 384, 520, True)
        out, scratch = torch.zeros(240, 384, device=DEV, dtype=torch.bfloat16), torch.empty(240, 768, device=DEV, dtype=torch.bfloat16)
        before = len(blaslt._ends)
        gemm.gated_nt(a[:, 1:513], w[:, 1:513], out, scratch, 200, "silu")
        assert len(blaslt._ends) == before
        want = _want(a[:200, 1:513], w[:, 1:513], 384, "gated")
        assert float((out[:200].double() - want).norm() / want.norm()) < 1e-2
    finally:
        blaslt.configure(plan_file=None)
        blaslt._plans.clear()
        blaslt._ends.clear()


@pytest.mark.parametrize("end", ["gated", "relu2", "add", "floats", None])
def test_a_tile_chosen_for_a_product_runs_it(tmp_path, monkeypatch, end):
    """Where tiles time faster, by measuring and then by another process's plan file: the tile runs, the result is right, and rows between the
    product's and the size it was chosen for are left alone."""
    from dinfer_amd.kernels import blaslt, gemm, ops
    m, n, k = 300, 512, 1024
    assert gemm.row_bucket(m) == 320
    ran = []
    tile = ops.gemm_tile

    def watched(a, w, out, rows, shape, **kw):
        ran.append((rows, shape, "gated" if kw.get("gated") else kw.get("act")))
        return tile(a, w, out, rows, shape, **kw)

    def timed(run):     # (a pass of its own has a product before it, which a tile may run)
        ran.clear()
        run()
        return 1.0 if ran and ran[-1][2] == (end if end in ("gated", "relu2") else None) else 2.0

    monkeypatch.setattr(ops, "gemm_tile", watched)

    monkeypatch.setattr(blaslt, "_least_of_three", lambda a, m, run: timed(run))
    monkeypatch.setattr(blaslt, "_in_trains", lambda w, forms, alone: [timed(lambda: form(w)) for form in forms])
    a, w = _inputs(m + 40, n, k, end == "gated", seed=4)
    scratch = torch.empty(m + 40, 2 * n, device=DEV, dtype=torch.bfloat16)
    start = torch.randn(m + 40, n, device=DEV).to(torch.bfloat16)

    def run():
        out = start.clone() if end == "add" else torch.full((m + 40, n), 7.0, device=DEV, dtype=torch.float32 if end == "floats" else torch.bfloat16)
        if end == "gated":
            gemm.gated_nt(a, w, out, scratch, m, "silu")
        elif end == "relu2":
            gemm.act_nt(a, w, out, m, "relu2")
        elif end == "add":
            assert gemm.add_nt(a, w, out, m)
        else:
            gemm.matmul_nt(a, w, out, m, may_pad=True)
        return out

    def forget():
        blaslt._plans.clear()
        blaslt._ends.clear()

    forget()
    blaslt.configure(tuning="measured", plan_file=str(tmp_path / "plans.json"))
    try:
        with blaslt.measuring():
            run()
        plans = lambda: [p for p in (*blaslt._plans.values(), *blaslt._ends.values()) if p and p.tile is not None]
        chosen = [p.tile.shape for p in plans()]
        assert chosen and any(e.get("tile") for e in json.loads((tmp_path / "plans.json").read_text()).values())
        forget()
        blaslt.configure(plan_file="")
        blaslt.configure(plan_file=str(tmp_path / "plans.json"))
        ran.clear()
        out = run()
        assert [r[:2] for r in ran] == [(m, plans()[0].tile.shape)] and [p.tile.shape for p in plans()] == chosen[-1:]
        assert all(p.times is None for p in plans())
        z = _want(a[:m], w, n, None if end == "floats" else end, start[:m])
        if end == "floats":
            torch.testing.assert_close(out[:m].double(), z, rtol=0, atol=4 * k ** 0.5 * 2.0 ** -24 * 8)    # (as above)
        else:
            _close(out[:m], z, str(end))
        assert torch.equal(out[m:], start[m:]) if end == "add" else bool((out[m:] == 7).all())
    finally:
        blaslt.configure(plan_file=None)
        forget()
