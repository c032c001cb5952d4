"""The products of the native step on their own: every tile shape with every epilogue, the
chained forms, and the few-row kernels by way of a one-layer step, against float64.

Tolerance of a product: the bf16 rounding of the result (8 significant bits: half an ulp is
up to 2^-8 of it), and for the fp32 sum of K products the bound K * 2^-24 * sum |x_i w_i| of
any order."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HALF_ULP = 2.0 ** -8
TILES = [(64, 64), (32, 128), (64, 128), (128, 128), (160, 128), (160, 128), (192, 128),
         (128, 256), (160, 256), (224, 256), (256, 256)]
CHAINS = {2: (4, 1), 3: (4, 2), 4: (2, 4)}


def _operands(seed, rows, outputs, reduction):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(rows, reduction, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(outputs, reduction, generator=g, device=DEV) * 0.05).to(torch.bfloat16)
    return x, w


def _exact(x, w):
    """The sums in float64 and how far any fp32 order can be from them."""
    xs, ws = x.double(), w.double()
    return xs @ ws.t(), x.shape[1] * 2.0 ** -24 * (xs.abs() @ ws.abs().t())


def _linear(x, w, out, form, tile):
    from nanovllm_jax_amd import _lib
    _lib.check(_lib.load().nvj_linear_launch(
        torch.cuda.current_stream().cuda_stream, x.data_ptr(), w.data_ptr(), out.data_ptr(),
        x.shape[0], w.shape[0], x.shape[1], form, tile), "nvj_linear_launch")


def _guarded(rows, columns):
    """An output with a row of ones before and behind it, which has to stay."""
    whole = torch.ones(rows + 2, columns, dtype=torch.bfloat16, device=DEV)
    return whole, whole[1:-1]


@pytest.mark.parametrize("tile", [-1] + list(range(len(TILES))))
@pytest.mark.parametrize("reduction", [64, 448])         # fewer steps than the ring, and more
def test_rows_of_every_tile(tile, reduction):
    print(f"case linear tile={tile} K={reduction}", flush=True)
    bm, bn = TILES[tile] if tile >= 0 else (128, 128)
    # one tile exactly, the edges of one, and several with a remainder in each direction
    for i, (rows, outputs) in enumerate([(bm, bn), (1, 8), (bm - 1, bn - 8), (bm + 1, bn + 8),
                                         (2 * bm + 5, 3 * bn + 24), (9 * bm + 3, bn)]):
        x, w = _operands(100 * tile + i, rows, outputs, reduction)
        want, bound = _exact(x, w)
        whole, out = _guarded(rows, outputs)
        _linear(x, w, out, 0, tile)
        err = (out.double() - want).abs()
        assert (err <= HALF_ULP * want.abs() + 1.01 * bound).all(), (rows, outputs)
        assert (whole[0] == 1).all() and (whole[-1] == 1).all()


@pytest.mark.parametrize("tile", [-1] + list(range(len(TILES))))
@pytest.mark.parametrize("rows,outputs", [(2048, 1024), (513, 4104), (1543, 8152), (1545, 8152)])
def test_rows_past_the_l2_of_every_tile(tile, rows, outputs):
    """4 to 24 MB of rows are stored by kernels of their own: both ends, and beyond."""
    print(f"case linear past L2 tile={tile} {rows} x {outputs}", flush=True)
    x, w = _operands(500 + tile + rows, rows, outputs, 128)
    want, bound = _exact(x, w)
    whole, out = _guarded(rows, outputs)
    _linear(x, w, out, 0, tile)
    err = (out.double() - want).abs()
    assert (err <= HALF_ULP * want.abs() + 1.01 * bound).all()
    assert (whole[0] == 1).all() and (whole[-1] == 1).all()


@pytest.mark.parametrize("tile", [-1] + list(range(len(TILES))))
def test_silu_mul_of_every_tile(tile):
    print(f"case linear silu tile={tile}", flush=True)
    bm, bn = TILES[tile] if tile >= 0 else (128, 128)
    for i, (rows, outputs) in enumerate([(bm, bn), (1, 32), (bm + 1, bn + 32),
                                         (2 * bm + 5, 3 * bn + 96)]):
        x, w = _operands(1000 + 100 * tile + i, rows, outputs, 320)
        sums, bound = _exact(x, w)
        half = outputs // 2
        g, u = sums[:, :half], sums[:, half:]
        sig = torch.sigmoid(g)
        want = g * sig * u
        # gate and up are bf16 values, up to half an ulp and the sums' error from g and u
        dg = HALF_ULP * g.abs() + 1.01 * bound[:, :half]
        du = HALF_ULP * u.abs() + 1.01 * bound[:, half:]
        slope = (sig * (1 + g * (1 - sig))).abs() + 0.25 * dg    # |silu''| < 1/2
        tol = slope * dg * (u.abs() + du) + (g * sig).abs() * du + 1.01 * HALF_ULP * want.abs()
        whole, out = _guarded(rows, half)
        _linear(x, w, out, 1, tile)
        assert ((out.double() - want).abs() <= tol).all(), (rows, outputs)
        assert (whole[0] == 1).all() and (whole[-1] == 1).all()


@pytest.mark.parametrize("form", CHAINS)
def test_chained_forms(form):
    print(f"case linear chains {CHAINS[form]}", flush=True)
    chains, run = CHAINS[form]
    unit = 32 * chains * run
    for i, (rows, outputs, reduction) in enumerate([
            (1, 8, unit), (32, 16, 2 * unit), (33, 24, 5 * unit), (17, 1000, 12 * unit),
            (128, 1024, 3072 // unit * unit), (97, 40, 7 * unit)]):
        x, w = _operands(2000 + 10 * form + i, rows, outputs, reduction)
        want, bound = _exact(x, w)
        whole, out = _guarded(rows, outputs)
        _linear(x, w, out, form, -1)
        err = (out.double() - want).abs()
        assert (err <= HALF_ULP * want.abs() + 1.01 * bound).all(), (rows, outputs, reduction)
        assert (whole[0] == 1).all() and (whole[-1] == 1).all()


def test_a_row_does_not_depend_on_the_rows_beside_it():
    """One order of the sums whatever the tile: the same bits from every shape, alone or in a
    batch."""
    print("case linear rows alone and together", flush=True)
    x, w = _operands(7, 300, 512, 1024)
    outs = []
    for tile in range(-1, len(TILES)):
        out = torch.empty(300, 512, dtype=torch.bfloat16, device=DEV)
        _linear(x, w, out, 0, tile)
        outs.append(out)
    assert all(torch.equal(o, outs[0]) for o in outs)
    for rows in (1, 31, 130):
        out = torch.empty(rows, 512, dtype=torch.bfloat16, device=DEV)
        _linear(x[100:100 + rows].contiguous(), w, out, 0, -1)
        assert torch.equal(out, outs[0][100:100 + rows])


@pytest.mark.parametrize("tile", [-1] + list(range(1, len(TILES))))
@pytest.mark.parametrize("norms,keep", [(True, True), (False, False)])
def test_qkv_projection_of_every_tile(tile, norms, keep):
    """Against the product alone and the rows launch on it, which is tested against the
    oracle: the same bits, with skipped and dropped slots, K and V kept or not."""
    print(f"case qkv linear tile={tile} norms={norms}", flush=True)
    from nanovllm_jax_amd import _lib
    lib = _lib.load()
    bm, bn = TILES[tile] if tile >= 0 else (128, 128)
    hq, hkv = (6, 1) if bn == 256 else (3, 2)
    heads, reduction, slots_n = hq + 2 * hkv, 192, 700
    for rows in (1, bm, bm + 1, 2 * bm + 7):
        x, w = _operands(3000 + rows, rows, heads * 128, reduction)
        g = torch.Generator(device=DEV).manual_seed(rows)
        cos_sin = torch.randn(50, 128, generator=g, device=DEV)
        norm = [torch.randn(128, generator=g, device=DEV) for _ in range(2)] if norms else [None] * 2
        rng = np.random.default_rng(rows)
        pos = torch.from_numpy(rng.integers(-1, 52, rows).astype(np.int32)).to(DEV)   # clamped
        slots = rng.permutation(slots_n)[:rows].astype(np.int32)
        slots[::5], slots[3::7] = -1, slots_n
        slots = torch.from_numpy(slots).to(DEV)
        ptr = lambda t: t.data_ptr() if t is not None else None
        stream = torch.cuda.current_stream().cuda_stream

        def caches():
            return [torch.ones(slots_n, hkv, 128, dtype=torch.bfloat16, device=DEV)
                    for _ in range(2)]

        qkv = torch.empty(rows, heads * 128, dtype=torch.bfloat16, device=DEV)
        _linear(x, w, qkv, 0, -1)
        want_q = torch.empty(rows, hq * 128, dtype=torch.bfloat16, device=DEV)
        want_kv = [torch.empty(rows, hkv * 128, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        want_c = caches()
        _lib.check(lib.nvj_qk_norm_rope_rows_launch(
            stream, qkv.data_ptr(), heads * 128, pos.data_ptr(), cos_sin.data_ptr(), 50,
            ptr(norm[0]), ptr(norm[1]), 1e-6, slots.data_ptr(), want_c[0].data_ptr(),
            want_c[1].data_ptr(), want_q.data_ptr(), hq * 128, want_kv[0].data_ptr(),
            want_kv[1].data_ptr(), hkv * 128, rows, hq, hkv, 128, slots_n), "rows")
        q = torch.empty_like(want_q)
        kept = torch.full_like(qkv, 3.0)
        got_c = caches()
        _lib.check(lib.nvj_qkv_linear_launch(
            stream, x.data_ptr(), w.data_ptr(), rows, reduction, pos.data_ptr(),
            cos_sin.data_ptr(), 50, ptr(norm[0]), ptr(norm[1]), 1e-6, slots.data_ptr(),
            got_c[0].data_ptr(), got_c[1].data_ptr(), q.data_ptr(),
            kept.data_ptr() if keep else None, hq, hkv, slots_n, tile), "qkv")
        assert torch.equal(q, want_q), rows
        assert all(torch.equal(a, b) for a, b in zip(got_c, want_c)), rows
        if keep:
            assert (kept[:, :hq * 128] == 3).all()
            assert torch.equal(kept[:, hq * 128:], torch.cat(want_kv, dim=1)), rows


def _layer_in_float64(runner, ids, attn_out_of):
    """One layer and the head of a runner, rounded to bf16 where the step rounds."""
    bf = lambda t: t.to(torch.bfloat16).double()
    c, lw = runner.cfg, runner.layers[0]

    def norm(s):
        return bf(s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + c.rms_norm_eps))

    h = runner.embed[ids.long()].double()
    qkv = bf(norm(h) @ lw["qkv"].double().t())
    o = attn_out_of(qkv)
    s = bf(o @ lw["o"].double().t()) + h
    gate, up = bf(norm(s) @ lw["gate_up"].double().t()).chunk(2, dim=-1)
    act = bf(gate * torch.sigmoid(gate) * up)
    s = bf(act @ lw["down"].double().t()) + bf(s)
    return norm(s) @ runner.embed.double().t()


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 16, 17, 32, 70, 130])
@pytest.mark.parametrize("hidden,inter,heads", [(256, 256, 2), (512, 3072, 8), (1024, 2816, 24),
                                                (2048, 512, 4)])
def test_one_layer_step_against_float64(rows, hidden, inter, heads, monkeypatch):
    """All the products of a step, few rows and many, on sequences of one position: attention
    over one key is its V row, so that nothing but products and norms is in the way."""
    print(f"case one layer rows={rows} hidden={hidden} inter={inter}", flush=True)
    from nanovllm_jax_amd.engine import decode_step as ds
    kv = 2
    cfg = ds.DecodeModelConfig(num_layers=1, hidden_size=hidden, num_heads=heads, num_kv_heads=kv,
                               head_dim=128, intermediate_size=inter, vocab_size=1000,
                               max_position=64, block_size=32, num_kvcache_blocks=rows)
    monkeypatch.setattr(ds, "_native_step_pays", lambda *sizes: True)
    runner = ds.DecodeStepRunner(cfg, DEV, seed=rows)
    ids = [(37 * i + 5) % 1000 for i in range(rows)]
    inputs = runner.make_inputs(ids, [1] * rows, [[i] for i in range(rows)])
    got = runner._native_forward(*inputs)
    assert got is not None

    def attend(qkv):
        v = qkv.view(rows, heads + 2 * kv, 128)[:, heads + kv:]
        return v.repeat_interleave(heads // kv, dim=1).reshape(rows, heads * 128)

    want = _layer_in_float64(runner, inputs[0], attend)
    # half an ulp of the logits, and on the way values whose fp32 sum fell on the other side
    # of a rounding: no more than six stages of independent errors of half an ulp
    err = (got.double() - want).norm(dim=1) / want.norm(dim=1)
    print("relative error", err.max().item(), "bound", 6 ** 0.5 * HALF_ULP, flush=True)
    assert err.max().item() <= 6 ** 0.5 * HALF_ULP, err.max().item()
