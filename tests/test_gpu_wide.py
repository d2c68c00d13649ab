"""The wide MXFP4 x Q8_0 product (k_mx_wide) at the edges of its forms: rows of
one part and of two (45 blocks and 46), the blocks a wave is padded by, one and
two 32-entry tiles, second passes of one entry, every bias type, and rows with
E8M0 scales outside the MFMA's range in each part of a row.  Every group is
sent to it (threshold 1); every stage is checked against the oracle fed the
GPU's own upstream bits, the block sums' order apart (helpers.REL_TOL)."""
import numpy as np
import pytest

from fixtures import device_moe_layer, moe_batch_fixture, moe_batch_x
from helpers import bits

pytestmark = pytest.mark.gpu


def _layer_run(ctx, O, lay, batch):
    from test_gpu_moe import _run, check_stagewise, gemm_path

    keep, cfg, lw = device_moe_layer(lay)
    x = moe_batch_x(batch, lay["hidden"], "normal")
    with gemm_path(ctx, "gemm"):
        g = _run(ctx, cfg, lw, x, batch)
    sample = sorted({0, 1, 31, 32, 33, 63, 64, 65, batch - 1} & set(range(batch * lay["topk"])))
    check_stagewise(O, lay, x, batch, g, sample=sample)
    return g, (keep, cfg, lw, x)


@pytest.mark.parametrize("hidden,dim,batch,bias", [
    (32, 32, 1, -1), (32, 32, 65, 0), (256, 288, 32, 1), (768, 800, 33, 30), (1440, 1472, 64, 0), (1472, 1440, 65, 30),
    (2880, 96, 130, 1), (96, 2880, 97, -1), (2848, 2880, 31, 0)])
def test_wide_edges(gpu_ctx, O, hidden, dim, batch, bias):
    """One expert takes every token, so the groups are exactly `batch` entries."""
    _layer_run(gpu_ctx, O, moe_batch_fixture(hidden, dim, 1, 1, bias, "normal"), batch)


@pytest.mark.parametrize("hidden,dim", [(96, 64), (1504, 1504)])
def test_wide_special_scales(gpu_ctx, O, hidden, dim):
    """Scales 0, 3, 241 and 255 in the first and the last block of some gate,
    up and down rows: those rows keep the integer form's values."""
    lay = moe_batch_fixture(hidden, dim, 2, 1, 0, "normal")
    for name, rows, nb in (("gate", dim, hidden // 32), ("up", dim, hidden // 32), ("down", hidden, dim // 32)):
        w = lay[name] = lay[name].copy()
        w = w.reshape(2, rows, nb, 17)
        for i, e in enumerate((0, 3, 241)):
            w[:, 5 + 9 * i, 0, 0] = e
            w[:, 7 + 9 * i, nb - 1, 0] = e
    lay["down"].reshape(2, hidden, dim // 32, 17)[1, 40, 0, 0] = 255
    _layer_run(gpu_ctx, O, lay, 70)


@pytest.mark.parametrize("hidden,dim", [(2880, 96), (96, 1472)])
def test_wide_place_in_list(gpu_ctx, O, hidden, dim):
    """An entry's result does not depend on its place in the list: the same
    tokens alone, in a one-tile pass and in a two-tile pass, bit for bit."""
    import torch

    from test_gpu_moe import gemm_path

    lay = moe_batch_fixture(hidden, dim, 1, 1, 0, "normal")
    keep, cfg, lw = device_moe_layer(lay)
    x = moe_batch_x(100, hidden, "normal").reshape(100, hidden)
    outs = []
    with gemm_path(gpu_ctx, "gemm"):
        for sel in (np.arange(100), np.arange(80, 100), np.arange(99, 100)):
            xd = torch.from_numpy(np.ascontiguousarray(x[sel])).cuda()
            out = torch.empty(len(sel) * hidden, dtype=torch.float32, device="cuda")
            gpu_ctx.forward_moe_batch(cfg, lw, xd, out, len(sel))
            torch.cuda.synchronize()
            outs.append(out.cpu().numpy().reshape(-1, hidden))
    assert np.array_equal(bits(outs[0][80:]), bits(outs[1]))
    assert np.array_equal(bits(outs[0][99:]), bits(outs[2]))


@pytest.mark.parametrize("batch,topk,experts", [(17, 2, 8), (64, 4, 128), (1024, 4, 256), (1023, 4, 37), (4096, 1, 64)])
def test_pack_lists_order(gpu_ctx, O, batch, topk, experts):
    """Lists, counts and offsets of large and ragged batches equal the
    reference's push-at-head order (kSelWaves parts of the selections)."""
    lay = moe_batch_fixture(32, 32, experts, topk, -1, "normal")
    keep, cfg, lw = device_moe_layer(lay)
    rng = np.random.default_rng(batch + experts)
    lg = rng.standard_normal((batch, experts)).astype(np.float32)
    from test_gpu_moe import _run

    g = _run(gpu_ctx, cfg, lw, moe_batch_x(batch, 32, "normal"), batch, lg.reshape(-1))
    counts, offsets, lst, active = O.group(g["ids"], g["weights"], batch, topk, experts)
    assert np.array_equal(g["counts"], counts) and np.array_equal(g["offsets"], offsets)
    assert np.array_equal(g["list"][:offsets[-1]], lst)


@pytest.mark.parametrize("hidden,experts,batch", [(2880, 128, 771), (96, 37, 2053), (4128, 256, 385)])
def test_route_wide_bits(gpu_ctx, O, hidden, experts, batch):
    """The large-batch router (8 x 8 logits a wavefront, 384 workgroups and
    more) gives the reference's accumulation order bit for bit: ragged experts
    and tokens, and a trailing half chunk of 32 elements."""
    import torch

    import spt

    rng = np.random.default_rng(hidden + batch)
    w = rng.standard_normal((experts, hidden)).astype(np.float32)
    b = rng.standard_normal(experts).astype(np.float32)
    x = rng.standard_normal((batch, hidden)).astype(np.float32)
    wd, bd, xd = (torch.from_numpy(v).cuda() for v in (w, b, x))
    t = spt.Tensor.make("ffn_gate_inp.weight", spt.TYPE_F32, [hidden, experts], wd.data_ptr(), w.nbytes)
    tb = spt.Tensor.make("ffn_gate_inp.bias", spt.TYPE_F32, [experts], bd.data_ptr(), b.nbytes)
    out = torch.empty(batch * experts, dtype=torch.float32, device="cuda")
    gpu_ctx.route_moe_batch(t, tb, xd, batch, out)
    torch.cuda.synchronize()
    rows = sorted({0, 1, 7, 8, 15, 16, batch // 2, batch - 2, batch - 1})
    want = O.route(w.reshape(-1), b, np.ascontiguousarray(x[rows]).reshape(-1), len(rows), hidden, experts)
    got = out.cpu().numpy().reshape(batch, experts)[rows]
    assert np.array_equal(bits(got.reshape(-1)), bits(np.asarray(want, np.float32).reshape(-1)))


@pytest.mark.parametrize("hidden,dim", [(128, 160), (256, 288), (384, 416), (512, 544), (640, 672),
                                        (768, 800), (1024, 1056), (1280, 1312),
                                        (1472, 1536), (1568, 2048), (2080, 2560), (2592, 64)])
def test_wide_forms(gpu_ctx, O, hidden, dim):
    """The row lengths at which a wave's blocks per part, and the loads of a
    stage, step up: 4 / 5, 8 / 9, 12 / 13, 16 / 17, 20 / 21 (two row tiles a step
    below, odd numbers of them too), 24 / 25, 32 / 33, 40 / 41 blocks in one
    part, 46, 48 / 49, 64 / 65, 80 / 81 in two; passes of two tiles and of one
    entry."""
    _layer_run(gpu_ctx, O, moe_batch_fixture(hidden, dim, 1, 1, 0, "normal"), 65)
