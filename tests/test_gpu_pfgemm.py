"""GPU prefill dequant-GEMMs (pf_gemm3 family) against the oracle.

Tolerance: norm-wise relative error <= 1e-3 per output row against the exact float64 product
of the fp16-dequantized weights and the fp16 activations, followed by the kernel's epilogue
(the RES epilogue is checked on out32 - res as well, so a large residual cannot hide an error
in the product).  Full-size launches (config 4, M = 2048) are checked on seeded weight-row
samples over every activation row.
"""
import numpy as np
import pytest
import torch

from oracle import gemv, quants
from thunderllamax_amd import formats, ops, synth
from thunderllamax_amd._lib import LAYOUT_PACKED, TlxError

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _iq3(rng, rows, kdim, dev):
    """Packed rows (what the oracle dequantizes) and their packed7 units on the GPU."""
    packed = formats.iq3_pack_rows(synth.iq3xxs_raw(rng, rows, kdim), kdim)
    return packed, torch.from_numpy(formats.iq3_pack7(packed, kdim)).to(dev)


def _rows_err(y, ref):
    return max(gemv.rel_err(y[m], ref[m]) for m in range(ref.shape[0]))


@pytest.mark.parametrize("M,N,K", [(256, 128, 512), (512, 256, 1024), (256, 384, 5120)])
def test_pfg3_ffn_parity(gpu, M, N, K):
    print(f"[case] pfg3_ffn M={M} N={N} K={K}", flush=True)
    rng = synth.config_rng(4)
    pg, wg = _iq3(rng, N, K, gpu)
    pu, wu = _iq3(rng, N, K, gpu)
    x = synth.activations_f16(rng, M, K)
    out = torch.empty(M, N, dtype=torch.float16, device=gpu)
    ops.pfg3_ffn(wg, wu, formats.gridf_tensor(gpu), torch.from_numpy(x).to(gpu), out)
    torch.cuda.synchronize()
    _, _, ref = gemv.pf_ffn_ref(quants.dequant_iq3xxs_packed(pg, K), quants.dequant_iq3xxs_packed(pu, K), x)
    err = _rows_err(out.cpu().numpy(), ref)
    print(f"[pfg3_ffn M={M} N={N} K={K}] max row rel-err {err:.3e}")
    assert err <= TOL


@pytest.mark.parametrize("M,N,K", [(256, 256, 512), (512, 512, 2048), (256, 256, 6144), (256, 256, 768)])
def test_pfg3_iq3o_parity(gpu, M, N, K):
    print(f"[case] pfg3_iq3o M={M} N={N} K={K}", flush=True)
    rng = synth.config_rng(4)
    pw, w = _iq3(rng, N, K, gpu)
    x = synth.activations_f16(rng, M, K)
    out = torch.empty(M, N, dtype=torch.float16, device=gpu)
    ops.pfg3_iq3o(w, formats.gridf_tensor(gpu), torch.from_numpy(x).to(gpu), out)
    torch.cuda.synchronize()
    _, ref = gemv.pf_o_ref(quants.dequant_iq3xxs_packed(pw, K), x)
    err = _rows_err(out.cpu().numpy(), ref)
    print(f"[pfg3_iq3o M={M} N={N} K={K}] max row rel-err {err:.3e}")
    assert err <= TOL


@pytest.mark.parametrize("M,N,K", [(256, 256, 512), (512, 512, 3072)])
def test_pfg3_iq3d_parity(gpu, M, N, K):
    print(f"[case] pfg3_iq3d M={M} N={N} K={K}", flush=True)
    rng = synth.config_rng(4)
    pw, w = _iq3(rng, N, K, gpu)
    x = synth.activations_f16(rng, M, K)
    res = rng.standard_normal((M, N)).astype(np.float32)
    out = torch.empty(M, N, dtype=torch.float32, device=gpu)
    ops.pfg3_iq3d(w, formats.gridf_tensor(gpu), torch.from_numpy(x).to(gpu), torch.from_numpy(res).to(gpu), out)
    torch.cuda.synchronize()
    acc, ref = gemv.pf_res_ref(quants.dequant_iq3xxs_packed(pw, K), x, res)
    y = out.cpu().numpy()
    err = _rows_err(y, ref)
    err_acc = _rows_err(y.astype(np.float64) - res, acc)
    print(f"[pfg3_iq3d M={M} N={N} K={K}] rel-err out {err:.3e}, product {err_acc:.3e}")
    assert err <= TOL and err_acc <= TOL


def test_pfg3_ffn_full_size_sampled_rows(gpu):
    """Config 4 gate+up: M=2048, K=5120, N=17408; 256 seeded weight rows over all 2048 rows."""
    print("[case] pfg3_ffn full-size M=2048", flush=True)
    rng = synth.config_rng(4)
    M, N, K = 2048, 17408, 5120
    pg, wg = _iq3(rng, N, K, gpu)
    pu, wu = _iq3(rng, N, K, gpu)
    x = synth.activations_f16(rng, M, K)
    out = torch.empty(M, N, dtype=torch.float16, device=gpu)
    ops.pfg3_ffn(wg, wu, formats.gridf_tensor(gpu), torch.from_numpy(x).to(gpu), out)
    torch.cuda.synchronize()
    cols = np.sort(np.random.default_rng(3).choice(N, 256, replace=False))
    _, _, ref = gemv.pf_ffn_ref(quants.dequant_iq3xxs_packed(pg[cols], K),
                                quants.dequant_iq3xxs_packed(pu[cols], K), x)
    y = out.cpu().numpy()[:, cols]
    err = _rows_err(y, ref)
    print(f"[pfg3_ffn full] max row rel-err {err:.3e}")
    assert err <= TOL
    assert np.isfinite(out.float().cpu().numpy()).all()


def test_pfg3_iq3d_full_size_sampled_rows(gpu):
    """Config 4 down: M=2048, K=17408, N=5120; 128 seeded weight rows over all 2048 rows."""
    print("[case] pfg3_iq3d full-size M=2048", flush=True)
    rng = synth.config_rng(4)
    M, N, K = 2048, 5120, 17408
    pw, w = _iq3(rng, N, K, gpu)
    x = synth.activations_f16(rng, M, K)
    res = rng.standard_normal((M, N)).astype(np.float32)
    out = torch.empty(M, N, dtype=torch.float32, device=gpu)
    ops.pfg3_iq3d(w, formats.gridf_tensor(gpu), torch.from_numpy(x).to(gpu), torch.from_numpy(res).to(gpu), out)
    torch.cuda.synchronize()
    cols = np.sort(np.random.default_rng(5).choice(N, 128, replace=False))
    acc, ref = gemv.pf_res_ref(quants.dequant_iq3xxs_packed(pw[cols], K), x, res[:, cols])
    y = out.cpu().numpy()[:, cols]
    err = _rows_err(y.astype(np.float64) - res[:, cols], acc)
    print(f"[pfg3_iq3d full] max row rel-err (product) {err:.3e}")
    assert err <= TOL


def test_pfg3_deterministic(gpu):
    """Two launches on the same inputs give identical bits (fixed k order, no atomics)."""
    print("[case] pfg3_iq3o determinism", flush=True)
    rng = synth.config_rng(4)
    M, N, K = 512, 512, 2048
    _, w = _iq3(rng, N, K, gpu)
    x = torch.from_numpy(synth.activations_f16(rng, M, K)).to(gpu)
    g = formats.gridf_tensor(gpu)
    a = torch.empty(M, N, dtype=torch.float16, device=gpu)
    b = torch.empty_like(a)
    ops.pfg3_iq3o(w, g, x, a)
    ops.pfg3_iq3o(w, g, x, b)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_pfg3_bad_arguments_raise(gpu):
    print("[case] pfg3 argument checks", flush=True)
    rng = synth.config_rng(4)
    g = formats.gridf_tensor(gpu)
    _, w = _iq3(rng, 256, 512, gpu)
    x = torch.zeros(256, 512, dtype=torch.float16, device=gpu)
    out = torch.empty(256, 256, dtype=torch.float16, device=gpu)
    with pytest.raises(TlxError):   # M not a multiple of 256
        ops.pfg3_iq3o(w, g, x[:128], out[:128])
    with pytest.raises(TlxError):   # only the packed7 layout is accepted
        ops.pfg3_iq3o(w, g, x, out, layout=LAYOUT_PACKED)
    with pytest.raises(TlxError):   # K not a multiple of 128
        ops.pfg3_iq3o(w, g, torch.zeros(256, 320, dtype=torch.float16, device=gpu), out)
    with pytest.raises(TlxError):   # N not a multiple of the 256-row tile
        ops.pfg3_iq3o(w, g, x, torch.empty(256, 128, dtype=torch.float16, device=gpu))


def _units(gpu, seed, rows, kdim):
    """packed7 units of seeded IQ3_XXS rows, repacked on the GPU."""
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    w = torch.randint(0, 256, (rows, 98 * (kdim // 256)), dtype=torch.uint8, device=gpu, generator=g)
    w[:, 96 * (kdim // 256):] = 0x14   # d (the packed rows' last field): fp16 1.22e-3
    return ops.pack_w7(w, torch.empty(rows * kdim // 2, dtype=torch.uint8, device=gpu), rows, kdim)


def _parts_written(ws, mark):
    """256 KB slots of the workspace that no longer hold the mark."""
    return int((ws.view(torch.int32)[:ws.numel() // 4].view(-1, 1 << 16) != mark).any(dim=1).sum())


# On 256 compute units: r tiles of K / 128 chunks; `parts` is G where G ranges divide the tiles, else
# G + r - gcd(G, r) (one a range and tile).
@pytest.mark.parametrize("M,N,K,mib,parts", [
    (256, 5120, 17408, 128, 240),   # 20 tiles: ranges that divide a tile, 12 each
    (256, 5120, 17408, 60, 240),    # the same in just 240 slots
    (256, 5120, 17408, 20, 80),     # 80 slots: 4 each
    (256, 5120, 17408, 11, 40),     # 44 slots: 2 each
    (256, 5120, 17408, 8, 0),       # 32 slots: whole tiles
    (512, 256, 4096, 128, 16),      # 2 tiles of 32 chunks, at least 4 chunks a range
    (512, 256, 512, 128, 8),        # 2 tiles of 4 chunks: 4 ranges of a chunk each
    (256, 256, 256, 128, 0),        # one tile of 2 chunks: whole
    (1024, 5120, 2048, 128, 240),   # 80 tiles of 16 chunks: 2 or 3 ranges a tile cost the same
    (2048, 5120, 17408, 128, 384),  # 160 tiles in 256 ranges: two segments a workgroup
    (2048, 5120, 17408, 104, 384),  # the same in the 415 slots that it asks for
    (2048, 5120, 17408, 103, 0),    # one MiB less: whole tiles
    (2048, 5120, 2304, 128, 0),     # 160 tiles of 18 chunks: whole tiles cost less than a split
    (256, 17408 * 2, 5120, 128, 384),   # 136 tiles of 40 chunks: two segments a workgroup
    (2048, 2048, 17408, 64, 256),   # 64 tiles in 256 slots: 4 ranges a tile
])
def test_pfg3_split_ranges(gpu, M, N, K, mib, parts):
    """The split schedules against whole tiles (no workspace): the parts that the workspace's room
    allows, the same products in another fp32 order (at most K roundings of 2^-24 of the row's norm-wise
    sum: 1e-5 holds), every output written, and the same bits on every call."""
    print(f"[case] pfg3 split M={M} N={N} K={K} workspace {mib} MiB", flush=True)
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the parts are those of 256 compute units")
    grid = formats.gridf_tensor(gpu)
    g = torch.Generator(device=gpu)
    g.manual_seed(M + N + K)
    x = torch.randn(M, K, device=gpu, generator=g).half()
    res = torch.randn(M, N, device=gpu, generator=g)
    w = _units(gpu, 1, N, K)
    mark = 0x7FABCDEF
    outs = []
    try:
        for size in (0, mib << 20, mib << 20):
            _, ws = ops.attach_workspace(gpu, gemm_bytes=size)
            y = torch.full((M, N), float("nan"), device=gpu)
            ffn = torch.full((M, N // 2), float("nan"), dtype=torch.float16, device=gpu)
            written = []
            for call_ in (lambda: ops.pfg3_iq3d(w, grid, x, res, y),
                          lambda: ops.pfg3_ffn(w[:w.numel() // 2], w[w.numel() // 2:], grid, x, ffn)):
                if ws is not None:
                    ws.view(torch.int32).fill_(mark)
                call_()
                torch.cuda.synchronize()
                if ws is not None:
                    written.append(_parts_written(ws, mark))
            outs.append((y, ffn))
            assert written == ([parts, parts] if size else []), written
    finally:
        ops.attach_workspace(gpu)
    (whole, fw), (split, fs), (again, fa) = outs
    assert torch.equal(split, again) and torch.equal(fs.view(torch.int16), fa.view(torch.int16))
    err = ((split - whole).double().norm(dim=1) / (whole - res).double().norm(dim=1)).max().item()
    assert err <= 1e-5, err
    # the fp16 SwiGLU of sums that differ by 1e-5: a few outputs move by one fp16 rounding (2^-11)
    errf = ((fs.double() - fw.double()).norm() / fw.double().norm()).item()
    assert errf <= 2.0 ** -11, errf
