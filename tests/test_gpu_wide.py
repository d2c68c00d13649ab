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


@pytest.mark.parametrize("batch,topk,experts", [(2048, 4, 256), (4095, 2, 256), (8191, 1, 37), (8192, 1, 256), (2730, 3, 5),
                                                (512, 16, 16)])
@pytest.mark.parametrize("path", ["gemm", "gemv"])
def test_large_launch_sequence(gpu_ctx, O, batch, topk, experts, path):
    """Up to 8,192 selections in one launch sequence (lists of more than 64 KB of
    LDS): every token's output has the bits of calls of at most 4,096 selections
    (neither path's result depends on an entry's place), and a sample of them the
    oracle's values."""
    import torch

    from test_gpu_moe import assert_close, gemm_path

    H, D = 96, 64
    lay = moe_batch_fixture(H, D, experts, topk, 0, "normal")
    rng = np.random.default_rng(batch + experts)
    lay["router"] = rng.standard_normal(experts * H).astype(np.float32)
    keep, cfg, lw = device_moe_layer(lay)
    x = rng.standard_normal(batch * H).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    whole, parts = torch.full_like(xd, 5.0), torch.full_like(xd, 7.0)
    step = 4096 // topk
    with gemm_path(gpu_ctx, path):
        gpu_ctx.forward_moe_batch(cfg, lw, xd, whole, batch)
        for t in range(0, batch, step):
            n = min(step, batch - t)
            gpu_ctx.forward_moe_batch(cfg, lw, xd[t * H:(t + n) * H], parts[t * H:(t + n) * H], n)
        torch.cuda.synchronize()
    got = whole.cpu().numpy()
    assert np.array_equal(bits(got), bits(parts.cpu().numpy()))
    rows = np.unique(np.r_[0:16, rng.integers(0, batch, 64), batch - 16:batch])
    want = O.forward_moe_batch(lay, np.ascontiguousarray(x.reshape(batch, H)[rows]).reshape(-1), len(rows), q8=True, threads=8)
    assert_close(got.reshape(batch, H)[rows].reshape(-1), want, what="sample")


@pytest.mark.parametrize("off", [1, 3, 10, 15])
@pytest.mark.parametrize("hidden,dim", [(1472, 96), (96, 1472), (2880, 64)])
def test_wide_unaligned_experts(gpu_ctx, O, hidden, dim, off):
    """Expert matrices that begin `off` bytes past a 16-byte boundary give the
    bits of aligned ones (rows of one part and of two, gate, up and down)."""
    import torch

    import spt
    from test_gpu_moe import gemm_path

    lay = moe_batch_fixture(hidden, dim, 3, 2, 0, "normal")
    keep, cfg, lw = device_moe_layer(lay)
    x = torch.from_numpy(moe_batch_x(70, hidden, "normal")).cuda()
    outs = []
    for o in (0, off):
        for name, shape in (("gate", [hidden, dim, 3]), ("up", [hidden, dim, 3]), ("down", [dim, hidden, 3])):
            buf = torch.zeros(lay[name].size + 64, dtype=torch.uint8, device="cuda")
            buf[o:o + lay[name].size] = torch.from_numpy(lay[name]).cuda()
            keep[f"{name} {o}"] = buf
            setattr(lw, f"ffn_{name}_exps", spt.Tensor.make(name, spt.TYPE_MXFP4, shape, buf.data_ptr() + o, lay[name].size))
        out = torch.full((70 * hidden,), 9.0, device="cuda")
        with gemm_path(gpu_ctx, "gemm"):
            gpu_ctx.forward_moe_batch(cfg, lw, x, out, 70)
            torch.cuda.synchronize()
        outs.append(bits(out.cpu().numpy()))
    assert np.array_equal(outs[0], outs[1])


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


@pytest.mark.parametrize("hidden,dim", [(256, 512), (768, 800), (1024, 1056), (1280, 1312), (1472, 1536), (1568, 2048),
                                        (2080, 2560), (2592, 64)])
def test_wide_forms(gpu_ctx, O, hidden, dim):
    """The row lengths at which a wave's blocks per part, and the loads of a
    stage, step up: 8, 16, 24 / 25, 32 / 33, 40 / 41, 46 / 48 blocks in one part,
    49, 64 / 65, 80 / 81 in two; passes of two tiles and of one entry."""
    _layer_run(gpu_ctx, O, moe_batch_fixture(hidden, dim, 1, 1, 0, "normal"), 65)


@pytest.mark.parametrize("hidden,dim", [(256, 320), (320, 288), (352, 320), (384, 416), (512, 288), (544, 320), (640, 288),
                                        (672, 320), (768, 288), (288, 768)])
def test_wide_two_row_tiles(gpu_ctx, O, hidden, dim):
    """Steps of two row tiles (256 experts of five steps and more): blocks a wave
    stepping up at 8 / 9, 12 / 13, 16 / 17, 20 / 21 and 24, odd numbers of row
    tiles; groups of 65 entries (two tiles, then one entry), 40, and one each;
    scales outside the MFMA's range in either tile."""
    from test_gpu_moe import _run, check_stagewise, gemm_path

    lay = moe_batch_fixture(hidden, dim, 256, 1, 0, "normal")
    for name, rows, nb in (("gate", dim, hidden // 32), ("up", dim, hidden // 32), ("down", hidden, dim // 32)):
        w = lay[name] = lay[name].copy()
        w = w.reshape(256, rows, nb, 17)
        w[5, 3, 0, 0] = 255
        w[5, 41, nb - 1, 0] = 3
        w[9, rows - 2, nb // 2, 0] = 241
    keep, cfg, lw = device_moe_layer(lay)
    batch = 136
    x = moe_batch_x(batch, hidden, "normal")
    logits = np.zeros((batch, 256), np.float32)
    expert = np.r_[np.full(65, 5), np.full(40, 9), np.arange(20, 51)]
    logits[np.arange(batch), expert] = 1.0
    with gemm_path(gpu_ctx, "gemm"):
        g = _run(gpu_ctx, cfg, lw, x, batch, logits.reshape(-1))
    check_stagewise(O, lay, x, batch, g, logits, sample=[0, 1, 31, 32, 63, 64, 65, 96, 97, 104, 105, 135])


@pytest.mark.parametrize("hidden,experts,small,batch,route", [
    (64, 128, 0, 192, "gemv"), (1536, 128, 0, 128, "gemv both"), (2880, 24, 12, 128, "both"),
    (512, 8, 0, 200, "both wide"), (2880, 24, 8, 128, "wide")])
def test_default_route(gpu_ctx, hidden, experts, small, batch, route):
    """The default policy's three choices, told apart by their bits (the GEMV and
    the wide product add the blocks in different orders): a narrow layer, and one
    of four selections an expert, on the GEMV alone; large groups beside twelve
    of three selections on both; large groups alone, or beside eight such (less
    than the GEMV's own launches), on the wide product alone.  (With no group on
    one side of the threshold two settings are the same.)"""
    import torch

    import spt

    g = torch.Generator(device="cuda")
    g.manual_seed(hidden + small)
    lw = spt.MoELayer()
    keep = [torch.randn(experts * hidden, generator=g, device="cuda") * 0.02]
    lw.ffn_gate_inp = spt.Tensor.make("router", spt.TYPE_F32, [hidden, experts], keep[0].data_ptr(), experts * hidden * 4)
    for name in ("gate", "up", "down"):
        w = torch.randint(0, 256, (experts * hidden * hidden // 32, 17), generator=g, device="cuda", dtype=torch.uint8)
        w[:, 0] = 118 + w[:, 0] % 7
        keep.append(w)
        setattr(lw, f"ffn_{name}_exps", spt.Tensor.make(name, spt.TYPE_MXFP4, [hidden, hidden, experts], w.data_ptr(), w.numel()))
    cfg = spt.MoEConfig(hidden, hidden, experts, 4)
    t = torch.arange(batch, device="cuda")
    large = experts - small
    logits = torch.zeros(batch, experts, device="cuda")
    for j in range(4):
        e = (4 * t + j) % large
        if j == 0 and small:  # three tokens each for the last `small` experts
            e = torch.where(t < 3 * small, large + t % small, e)
        logits[t, e] = 1.0 + j
    x = torch.randn(batch * hidden, generator=g, device="cuda")
    outs = {}
    try:
        for name, threshold in (("default", 0), ("gemv", 1 << 30), ("both", 5), ("wide", 1)):
            gpu_ctx.set_gemm_min_group(threshold)
            outs[name] = torch.empty(batch * hidden, device="cuda")
            gpu_ctx.forward_moe_batch(cfg, lw, x, outs[name], batch, spt.make_taps(logits_in=logits))
            torch.cuda.synchronize()
    finally:
        gpu_ctx.set_gemm_min_group(0)
    same = [n for n in ("gemv", "both", "wide") if torch.equal(outs["default"].view(torch.int32), outs[n].view(torch.int32))]
    assert same == route.split()


@pytest.mark.parametrize("bias,off", [(0, 1), (0, 2), (0, 3), (1, 1), (30, 1)])
@pytest.mark.parametrize("form", ["arena", "noalloc"])
def test_wide_biases_between_elements(gpu_ctx, O, bias, off, form):
    """Expert biases that begin between elements give a forced wide product the
    same bits as aligned ones (and not the GEMV's, whose sums differ)."""
    import torch

    import spt
    from test_gpu_moe import gemm_path

    lay = moe_batch_fixture(768, 800, 3, 2, bias, "normal")
    keep, cfg, lw = device_moe_layer(lay)
    batch = 70
    x = torch.from_numpy(moe_batch_x(batch, 768, "normal")).cuda()

    def run(path):
        out = torch.full((batch * 768,), 9.0, device="cuda")
        with gemm_path(gpu_ctx, path):
            if form == "arena":
                gpu_ctx.forward_moe_batch(cfg, lw, x, out, batch)
            else:
                from test_zz_no_alloc import _noalloc

                assert _noalloc(gpu_ctx, cfg, lw, x, out, batch) == spt.OK
            torch.cuda.synchronize()
        return bits(out.cpu().numpy())

    want, gemv = run("gemm"), run("gemv")
    assert not np.array_equal(want, gemv)
    for name in ("gate_bias", "up_bias", "down_bias"):
        field = f"ffn_{name.split('_')[0]}_exps_bias"
        t = getattr(lw, field)
        buf = torch.zeros(t.nbytes + 8, dtype=torch.uint8, device="cuda")
        buf[off:off + t.nbytes] = keep[name].view(torch.uint8)
        keep["moved " + name] = buf
        shape = [t.shape[i] for i in range(t.n_dims)]
        setattr(lw, field, spt.Tensor.make(name, bias, shape, buf.data_ptr() + off, t.nbytes))
    assert np.array_equal(run("gemm"), want) and np.array_equal(run("gemv"), gemv)
