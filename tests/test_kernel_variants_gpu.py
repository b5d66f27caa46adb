"""GPU parity of single kernel variants and dispatch branches, at the sizes where each can go wrong."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def af3():
    import af3_kernels_amd
    af3_kernels_amd._lib.load()
    return af3_kernels_amd


def f32np(t):
    return t.detach().float().cpu().numpy()


@pytest.mark.parametrize("H,L,D,pad,first", [
    (1, 1, 24, 0, 0), (2, 2, 24, 1, 1), (3, 31, 32, 0, 1), (2, 33, 8, 3, 0), (1, 63, 24, 0, 0), (1, 65, 48, 0, 1),   # one wavefront, last tile nearly empty
    (2, 129, 24, 0, 0), (2, 190, 32, 5, 1), (3, 257, 24, 0, 0),   # key tiles split over four wavefronts
    (2, 129, 48, 0, 1), (2, 322, 64, 0, 0),                       # a pair of wavefronts per workgroup
    (16, 513, 48, 1, 0),                                          # two pairs, head_dim padded to 64
    (16, 515, 24, 1, 1),                                          # pairs on shared tiles, four computing wavefronts
    (16, 1027, 24, 0, 0), (16, 1024, 24, 7, 1),                   # ... eight
    (16, 1027, 48, 0, 1), (16, 1032, 40, 0, 0), (16, 1090, 48, 6, 0),   # eight, head_dim up to 48 padded to 64, P.V in its own stage
    (16, 1027, 56, 0, 1), (16, 1032, 64, 0, 0),                   # loading wavefronts, one query block each
    (16, 2051, 24, 0, 0), (16, 2050, 48, 1, 0),                   # four wavefronts that load for themselves
])
def test_single_row_bias_at_any_address(af3, oracle, H, L, D, pad, first):
    """One batch row, bias rows that start at any element: what surrounds the L x L corner (here NaN) must not be used."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    M = L + pad
    flat = torch.full((first + H * M * M,), float("nan")).to(torch.bfloat16)
    bias = flat[first:].view(H, M, M)
    bias[:, :L, :L] = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(L, generator=g) < 0.8
    keep[L // 2] = True
    dev = flat.cuda()[first:].view(H, M, M)
    print("case", H, L, D, pad, first, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), dev)
    torch.cuda.synchronize()
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias[:, :L, :L]))
    assert np.abs(f32np(out) - want).max() <= 2e-2


@pytest.mark.parametrize("rank", [None, 1, 2, 4, "float"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_native_host_path_equals_the_python_path(af3, dtype, rank):
    """Plain calls are prepared in native code, the rest (here: the implementation called directly, a mask that is not bool) in
    Python: same bits, whatever the mask's shape; strided q, k, v and a padded bias included."""
    from af3_kernels_amd import ops
    B, H, L, D = 3, 4, 72, 32
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B, L, H, D, generator=g).to(dtype).cuda().transpose(1, 2) for _ in range(3))
    bias = torch.randn(H, L + 8, L + 8, generator=g).to(dtype).cuda()
    keep = (torch.rand(B, L, generator=g) < 0.8).cuda()
    mask = {None: None, 1: keep[0], 2: keep, 4: keep[:, None, None, :], "float": keep.float()}[rank]
    got = af3.dot_product_attention_cpp(q, k, v, mask, bias)
    want = ops._dpa_forward_impl(q, k, v, ops._lift_mask(mask, L), bias, ops._DTYPE_CODE[dtype], False)
    assert got.shape == q.shape and torch.equal(got, want)


def test_native_host_path_follows_updated_weights(af3):
    """Matrices derived from weights are recomputed when a weight changes in place or is replaced."""
    from af3_kernels_amd import fused
    g = torch.Generator().manual_seed(4)
    n, C, head = 48, 128, 4
    x, mask, bias = torch.randn(n, C, generator=g).to(torch.bfloat16).cuda(), torch.ones(n, dtype=torch.bool).cuda(), torch.randn(head, n, n, generator=g).to(torch.bfloat16).cuda()
    ws = [af3.vnni_repack_tensor((torch.randn(C, C, generator=g) / C ** 0.5).to(torch.bfloat16).cuda(), 2, C // head) for _ in range(4)]
    qb = torch.randn(C, generator=g).to(torch.bfloat16).cuda()
    glu_w = (torch.randn(C, 2 * C, generator=g) / C ** 0.5).to(torch.bfloat16).cuda()

    def both():
        return af3.self_attention_cpp(x, mask, bias, ws[0], qb, ws[1], ws[2], ws[3], head), af3.gated_linear_unit_cpp(x, glu_w)

    first = both()
    assert all(torch.equal(a, b) for a, b in zip(first, both()))
    for change in (lambda: (ws[1].mul_(2), glu_w.mul_(2)), lambda: (ws.__setitem__(2, ws[2] * 2), qb.add_(1)), lambda: (qb.data.mul_(3), fused.clear_weight_cache())):
        before = both()
        change()
        after = both()
        assert not torch.equal(before[0], after[0])
        fused.clear_weight_cache()
        assert all(torch.equal(a, b) for a, b in zip(after, both()))
    assert not torch.equal(first[1], both()[1])


@pytest.mark.parametrize("B,H,L,D", [
    (1, 2, 97, 32), (2, 3, 130, 24), (1, 1, 1023, 32),       # four wavefronts per block of 32 query rows
    (5, 4, 385, 32), (16, 4, 255, 8),                        # ... two blocks per workgroup
    (16, 4, 385, 32), (64, 4, 97, 24),                       # two wavefronts per block, four blocks
    (3, 4, 161, 64), (9, 8, 250, 40),                        # head_dim padded to 64, two wavefronts per block
    (33, 8, 131, 32), (40, 8, 97, 64), (3, 2, 95, 20),       # one wavefront per block
])
@pytest.mark.parametrize("kind", ["random", "lopsided", "ramp", "far"])
def test_fp32_forms(af3, oracle, B, H, L, D, kind):
    """The fp32 kernel's launch forms; masks that leave wavefronts of a key split without a tile, logits that run away from the
    first tile's reference, references of extreme magnitude."""
    g = torch.Generator().manual_seed(B + L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g)
    keep = torch.rand(B, L, generator=g) < 0.8
    if kind == "lopsided":
        keep[:] = False
        keep[::2, : min(L, 40)] = True
        keep[1::2, L // 2] = True
        keep[B // 2] = False
    elif kind == "ramp":
        bias += torch.linspace(-60.0, 80.0, L)
    elif kind == "far":
        bias[:, ::3] -= 3.0e6
        bias[:, 1::3, : L // 2] = float("-inf")
    if kind != "lopsided":
        keep[:, L - 1] = True
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda())
    torch.cuda.synchronize()
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias))
    rows = slice(None) if kind != "far" else slice(1, None, 3)      # (an offset of 3e6 leaves a logit two bits behind the point)
    assert np.isfinite(f32np(out)).all()
    assert np.abs(f32np(out) - want)[:, :, rows].max() <= 2e-5
    if kind == "far":
        assert np.abs(f32np(out) - want).max() <= 0.5


@pytest.mark.parametrize("B,H,L,D,pad", [
    (37, 4, 37, 32, 0), (2, 1, 1, 8, 3), (3, 2, 129, 24, 1), (16, 4, 128, 32, 0),      # one round of workgroups
    (128, 4, 128, 32, 0), (125, 4, 127, 32, 1),                                        # 512 and 500 workgroups of 128 rows: the most that read in place
    (129, 4, 128, 32, 0), (129, 4, 127, 24, 0),                                        # 516: shared-bias kernel
    (5, 16, 191, 48, 0), (2, 16, 255, 64, 1), (48, 16, 70, 48, 0), (49, 16, 70, 48, 3),   # head_dim padded to 64; up to 768 workgroups, past it a workspace
    (40, 4, 200, 24, 5), (64, 4, 203, 32, 0),                                          # workspace written from rows at any address
])
def test_batched_bias_at_any_address(af3, oracle, B, H, L, D, pad):
    """Batches on both sides of the line up to which the one-row kernel reads the bias in place, and rewrites of ragged rows."""
    g = torch.Generator().manual_seed(B + L)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    M = L + pad
    bias = torch.full((H, M, M), float("nan")).to(torch.bfloat16)
    bias[:, :L, :L] = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g) < 0.8
    keep[:, L // 2] = True
    keep[B // 2] = False
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda())
    torch.cuda.synchronize()
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias[:, :L, :L]))
    assert np.abs(f32np(out) - want).max() <= 2e-2


@pytest.mark.parametrize("with_row", [True, False])
@pytest.mark.parametrize("M,N,K,form", [
    (1, 64, 64, 0), (65, 128, 64, 11), (63, 320, 192, 11), (129, 64, 128, 21), (200, 256, 320, 13), (64, 192, 64, 13), (257, 192, 256, 22),
    (127, 448, 64, 23), (129, 384, 448, 23), (1000, 1536, 384, 0), (2049, 3072, 768, 0),
])
def test_projection_forms(af3, M, N, K, form, with_row):
    """The projection product against the same product in float32, per tile form; rows behind M and columns behind N are not touched."""
    import ctypes
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w, row = (torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16) for s in ((M, K), (N, K), (N,)))
    out = torch.full((M + 1, N), 7.0, device="cuda", dtype=torch.bfloat16)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    print("case", M, N, K, form, with_row, flush=True)
    rc = af3._lib.load().af3_project(ptr(x), ptr(w), ptr(row) if with_row else None, ptr(out), ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(K), form,
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert rc == 0
    want = x.float() @ w.float().t() + (row.float() if with_row else 0.0)
    assert (out[:M].float() - want).abs().max() <= 2 ** -8 * want.abs().max()
    assert bool((out[M] == 7.0).all())


@pytest.mark.parametrize("B,H,L,D", [(1, 1, 1, 8), (1, 2, 3, 24), (2, 1, 4, 40), (1, 2, 63, 16), (1, 1, 257, 32), (2, 1, 1026, 24), (1, 1, 4161, 24), (1, 1, 8192, 24),
                                     (66, 8, 130, 24), (17, 8, 450, 16), (6, 16, 705, 32), (3, 16, 770, 48)])   # launches of many workgroups: keys not in parts
@pytest.mark.parametrize("kind", ["random", "first", "last", "one tile", "none", "bytes", "no mask"])
def test_fp8_mask_rows(af3, B, H, L, D, kind):
    """Mask rows shorter than one load, ending inside a load, of more than 64 tiles; rows with one live key or none; keep bytes other than 1."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16).cuda() for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16).cuda()
    keep = torch.rand(L + 1, generator=g)[1:] < 0.8
    if kind in ("first", "last", "one tile", "none"):
        keep[:] = False
        keep[{"first": slice(0, 1), "last": slice(L - 1, L), "one tile": slice(L // 2, L // 2 + 3), "none": slice(0, 0)}[kind]] = True
    dev = keep.to(torch.uint8).mul(0x80).cuda().view(torch.bool) if kind == "bytes" else keep.cuda()
    print("case", B, H, L, D, kind, flush=True)
    out = af3.dot_product_attention_fp8(q, k, v, None if kind == "no mask" else dev, bias)
    torch.cuda.synchronize()
    keep = torch.ones(L, dtype=torch.bool) if kind == "no mask" else keep
    vd, vs = af3.quantize_fp8_e4m3(v)
    s = (q.float() * D ** -0.5).matmul(k.float().transpose(-1, -2).contiguous()) + bias.float()
    p = (s.masked_fill(~keep.cuda(), float("-inf")) if keep.any() else torch.zeros_like(s)).softmax(-1)
    # e4m3 weights: each within 2^-4 of itself, as in the test of the bias forms
    bound = 2 ** -4 * p.matmul((vd.float() * vs).abs()) + 2e-2
    assert bool(((out.float() - p.matmul(vd.float() * vs)).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,L,D", [(1, 1, 1, 8), (1, 1, 5, 8), (1, 3, 77, 24), (2, 16, 515, 24), (3, 16, 1536, 24), (5, 16, 1541, 24), (5, 16, 1536, 32)])   # up to more than four loads per thread
def test_fp8_scale_sees_every_element(af3, B, H, L, D, dtype):
    """One large element of v anywhere: a maximum that missed it would clamp it.  With q = 0 and no bias the output is the mean of v, here 2^10 / L."""
    q, k = torch.zeros(B, H, L, D, dtype=dtype, device="cuda"), torch.ones(B, H, L, D, dtype=dtype, device="cuda")
    n = q.numel()
    for at in sorted({0, n - 1, n // 2, n - 9 if n > 9 else 0, (1 << 19) % n, min(n - 1, 3 * (1 << 19) + 5)}):
        v = torch.zeros(n, dtype=dtype, device="cuda")
        v[at] = 1024.0
        print("case", B, H, L, D, at, flush=True)
        out = af3.dot_product_attention_fp8(q, k, v.view(B, H, L, D), None, None)
        b, h, d = at // (H * L * D), at // (L * D) % H, at % D
        want = torch.zeros(B, H, 1, D, device="cuda")
        want[b, h, 0, d] = 1024.0 / L
        assert bool(((out.float() - want).abs() <= 2 ** -8 * want).all())


@pytest.mark.parametrize("B,H,L,D", [(2, 64, 20, 24), (3, 33, 130, 24), (2, 9, 1000, 16), (5, 16, 512, 32), (7, 13, 641, 48)])   # from 64 blocks of 128 rows on, numbers of them that 8 does not divide
def test_fp8_batch_rows_side_by_side(af3, B, H, L, D):
    """Workgroups dealt by blocks of query rows compute what those of single batch rows do, dealt by heads and perhaps with the keys in parts (whose
    maxima differ, and with them the roundings of the e4m3 weights)."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).clamp(-3.9, 3.9).to(torch.bfloat16).cuda() for _ in range(3))
    for t in (q, k, v):
        t[:, 0, 0, 0] = 4.0   # (one scale for every batch row)
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16).cuda()
    keep = (torch.rand(L, generator=g) < 0.8).cuda()
    print("case", B, H, L, D, flush=True)
    out = af3.dot_product_attention_fp8(q, k, v, keep, bias)
    # independent weight errors of at most 2^-4 on each side: sum p v e has at most 2^-4 of the rms of sum p v for random v, twice that for both
    # (a block in the wrong place: 2^0.5 of it)
    for b in range(B):
        one = af3.dot_product_attention_fp8(q[b:b + 1], k[b:b + 1], v[b:b + 1], keep, bias).float()
        for i in range(0, L, 128):
            assert (out[b:b + 1, :, i:i + 128].float() - one[:, :, i:i + 128]).norm() <= 2 ** -3 * one[:, :, i:i + 128].norm()


@pytest.mark.parametrize("compensated", [True, False])
@pytest.mark.parametrize("B,H,L,D,mask_kind", [
    (1, 1, 1, 24, "none"), (2, 3, 33, 24, "random"), (1, 2, 64, 32, "none"), (2, 2, 65, 16, "tail"), (3, 2, 127, 48, "random"), (1, 3, 128, 64, "tail"),
    (5, 2, 200, 24, "late"), (2, 4, 259, 24, "random"), (1, 2, 321, 56, "late"), (2, 16, 512, 24, "tail"), (1, 16, 1027, 24, "random"),
])
def test_fp8_bias_forms_and_tile_flags(af3, B, H, L, D, mask_kind, compensated):
    """Bias rows at any address, tiles with and without dropped keys, leading tiles without a live key: the kernel against the formula on the
    dequantised operands (for the compensated product: on q and k themselves)."""
    g = torch.Generator().manual_seed(L + D + B)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16).cuda() for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16).cuda()
    keep = {"none": torch.ones(L), "random": (torch.rand(L, generator=g) < 0.8).float(), "tail": (torch.arange(L) < L - L // 10).float(), "late": (torch.arange(L) >= L * 5 // 8).float()}[mask_kind].bool()
    keep[L - 1] = True
    print("case", B, H, L, D, mask_kind, compensated, flush=True)
    out = af3.dot_product_attention_fp8(q, k, v, keep.cuda(), bias, compensated=compensated)
    torch.cuda.synchronize()
    vd, vs = af3.quantize_fp8_e4m3(v)
    qq, kk = q.float() * D ** -0.5, k.float()
    if not compensated:
        (q8, qs), (k8, ks) = af3.quantize_fp8_e4m3(q, D ** -0.5), af3.quantize_fp8_e4m3(k)
        qq, kk = q8.float() * qs, k8.float() * ks
    s = qq.matmul(kk.transpose(-1, -2)) + bias.float()
    p = s.masked_fill(~keep.cuda(), float("-inf")).softmax(-1)
    want = p.matmul(vd.float() * vs)
    # e4m3 weights: each within 2^-4 of itself
    bound = 2 ** -4 * p.matmul((vd.float() * vs).abs()) + 2e-2
    assert bool(((out.float() - want).abs() <= bound).all())


def grid_block_case(af3, N, transpose):
    """(module, pair, mask, its result in float32 with bf16 roundings where the block stores bf16)"""
    g = torch.Generator(device="cuda").manual_seed(N)
    mod = af3.GridSelfAttentionCpp(128, 4, transpose).to("cuda", torch.bfloat16).eval().requires_grad_(False)
    for name, p in mod.named_parameters():
        p.copy_(torch.randn(p.shape, generator=g, device="cuda") * (128 ** -0.5 if p.dim() == 2 else 0.1) + (1.0 if name == "act_norm.weight" else 0.0))
    pair = torch.randn(N, N, 128, generator=g, device="cuda").mul_(2.0).add_(0.5).to(torch.bfloat16)
    keep = torch.rand(N, N, generator=g, device="cuda") < 0.8
    keep[:, 0] = True
    if N > 2:
        keep[1] = False   # a row without any live key
    bf = lambda t: t.to(torch.bfloat16).float()
    f = lambda m: m.weight.float()
    x = bf(torch.nn.functional.layer_norm(pair.float(), (128,), f(mod.act_norm), mod.act_norm.bias.float(), mod.act_norm.eps))
    bias = bf(torch.nn.functional.linear(x, f(mod.pair_bias_projection))).permute(2, 0, 1)
    rows = x.transpose(0, 1) if transpose else x
    q, k, v, gate = (torch.nn.functional.linear(rows, f(m)).view(N, N, 4, 32).transpose(1, 2).contiguous()
                     for m in (mod.q_projection, mod.k_projection, mod.v_projection, mod.gating_query))
    s = bf(q * 32 ** -0.5).matmul(bf(k).transpose(-1, -2).contiguous()) + bias
    s = s.masked_fill(~keep[:, None, None, :], -1e9)
    o = s.softmax(-1).matmul(bf(v)) * torch.sigmoid(bf(gate))
    want = torch.nn.functional.linear(bf(o.transpose(1, 2).reshape(N, N, 128)), f(mod.output_projection))
    if transpose:
        want = want.transpose(0, 1)
    return mod, pair, keep, want


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("N", [1, 2, 31, 33, 64, 97, 150, 161, 200, 229, 330])
def test_grid_block_projected_form(af3, N, transpose):
    """The grid block (projections in one pass, attention, output projection) against the same steps in float32, with bf16 roundings where
    the block stores bf16: partial token blocks, heads in separate workgroups and together, query tiles with idle wavefronts, gate rows of one to
    four batch rows, both orientations."""
    mod, pair, keep, want = grid_block_case(af3, N, transpose)
    print("case", N, transpose, flush=True)
    out = mod(pair, keep)
    again = mod(pair, keep)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    err = (out.float() - want).abs()
    assert err.max() <= 3e-2 * max(1.0, float(want.abs().max())) and err.norm() <= 1e-2 * want.norm()


@pytest.mark.parametrize("N,transpose", [(737, False), (700, True)])
def test_grid_block_where_memory_is_short(af3, N, transpose):
    """The projections of the whole call take four times the pair tensor; where that is not there the block runs in slabs of batch
    rows, in the memory of a result, a slab of 256 MB, its gated rows and a bias, with room for a rewritten bias."""
    mod, pair, keep, want = grid_block_case(af3, N, transpose)
    free = mod(pair, keep)
    need = N * N * (256 + 8) + (256 << 20) * 5 // 4 + 4 * 4 * 768 ** 2 + (24 << 20)
    assert need < N * N * (5 * 256 + 8)
    want, free = want.cpu(), free.cpu()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    print("case", N, transpose, flush=True)
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + need) / total)
    try:
        out = mod(pair, keep).cpu()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    err = (out.float() - want).abs()
    assert err.max() <= 3e-2 * max(1.0, float(want.abs().max())) and err.norm() <= 1e-2 * want.norm()
    assert (out.float() - free.float()).norm() <= 4e-3 * want.norm()


@pytest.mark.parametrize("M,K,N", [(1, 64, 32), (33, 128, 480), (65, 64, 544), (524289 + 31, 64, 256), (262145, 128, 544)])
def test_glu_whole_row_stores(af3, M, K, N):
    """Outputs narrower and wider than a workgroup's 512 columns, partial blocks of rows, and outputs beyond 256 MB (their stores bypass the caches)."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(K, 2 * N, generator=g, device="cuda", dtype=torch.bfloat16) * K ** -0.5
    print("case", M, K, N, flush=True)
    out = af3.gated_linear_unit_cpp(x, w)
    torch.cuda.synchronize()
    for rows in (slice(0, 4096), slice(max(0, M - 4096), M), slice(M // 2, M // 2 + 4096)):
        a, b = (x[rows].float() @ w.float()).chunk(2, dim=-1)
        want = torch.nn.functional.silu(a) * b
        assert (out[rows].float() - want).abs().max() <= 2 ** -7 * want.abs().max()


FP32_FORMS = [(1, 2, 97, 32), (5, 4, 385, 32), (16, 4, 385, 32), (3, 4, 161, 64), (33, 8, 131, 32), (40, 8, 97, 64), (3, 2, 95, 20)]   # (every launch form of the fp32 kernel)


@pytest.mark.parametrize("B,H,L,D", FP32_FORMS)
@pytest.mark.parametrize("garbage", [1e10, -1e10, 1e30, float("inf"), float("nan")])
def test_fp32_dropped_keys_are_replaced_whatever_they_hold(af3, oracle, B, H, L, D, garbage):
    """masked_fill replaces the finished logit of a dropped key: what K holds there has no weight, in tiles with and without live
    keys; a batch row without any live key is the mean of V."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g)
    keep = torch.rand(B, L, generator=g) < 0.7
    keep[:, L - 1] = True
    keep[0, 40:70] = False
    if B > 1:
        keep[1] = False
    dirty = torch.where(keep[:, None, :, None], k, torch.tensor(garbage))
    out = af3.dot_product_attention_cpp(q.cuda(), dirty.cuda(), v.cuda(), keep.cuda(), bias.cuda())
    torch.cuda.synchronize()
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias))
    assert np.abs(f32np(out) - want).max() <= 2e-5


@pytest.mark.parametrize("B,H,L,D", [(4, 4, 300, 64), (16, 4, 200, 32), (24, 8, 300, 64), (2, 4, 768, 32)])
@pytest.mark.parametrize("kind,bound", [("wide", 3e-7), ("ramp", 5e-7)])
def test_fp32_biases_join_finished_products(af3, B, H, L, D, kind, bound):
    """Wide biases and biases that grow along the row keep the precision of one rounding per bias: relative 2-norm errors against 64 bits of
    1.6e-7 to 2.5e-7 and 2.1e-7 to 4.3e-7 (a kernel of fp32 matrix instructions: 2.2e-7 to 2.8e-7 and 3.9e-7 to 4.7e-7; products accumulated on
    top of bias minus reference, rounded at that magnitude up to 24 times: 4.0e-7 and up to 1.8e-6)."""
    g = torch.Generator(device="cuda").manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g, device="cuda") for _ in range(3))
    bias = torch.randn(H, L, L, generator=g, device="cuda")
    bias = bias * 10 if kind == "wide" else bias + torch.linspace(-20, 20, L, device="cuda")
    keep = torch.rand(B, L, generator=g, device="cuda") < 0.92
    keep[:, 0] = True
    out = af3.dot_product_attention_cpp(q, k, v, keep, bias)
    torch.cuda.synchronize()
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * D ** -0.5 + bias.double()
    want = s.masked_fill(~keep[:, None, None, :], -1e9).softmax(-1) @ v.double()
    assert (out.double() - want).norm() <= bound * want.norm()


@pytest.mark.parametrize("B,H,L,D", FP32_FORMS)
@pytest.mark.parametrize("kind", ["k+inf", "k-inf", "k nan", "q inf", "v+inf", "v both", "v huge", "v ramp", "bias+inf"])
def test_fp32_infinities_act_as_in_the_formula(af3, B, H, L, D, kind):
    """Infinities and NaN of live keys: the logit or sum they make in the formula, NaN rows where that has NaN, every other row and
    column as without them.  Finite values beyond bf16's largest, and sums that only overflow under a reference left behind, stay finite."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g)
    keep = torch.rand(B, L, generator=g) < 0.8
    j, j2 = L // 2, L - 1                       # keys of two tiles, both live
    keep[:, [j, j2]] = True
    inf, b, h = float("inf"), B - 1, H - 1
    if kind[0] == "k":
        k[b, h, j, 1] = {"k+inf": inf, "k-inf": -inf, "k nan": float("nan")}[kind]
    elif kind == "q inf":
        q[b, h, 3, 2] = inf
    elif kind == "bias+inf":
        bias[h, 5, j] = inf
    elif kind == "v ramp":
        v *= 1e35
        bias += torch.linspace(0.0, 20.0, L)
    else:
        v[b, h, j, 1] = inf if kind != "v huge" else 3.4e38
        if kind == "v both":
            v[b, h, j2, 1] = -inf
    print("case", B, H, L, D, kind, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()).cpu()
    s = (q.double() @ k.double().transpose(-1, -2)) * D ** -0.5 + bias.double()
    want = s.masked_fill(~keep[:, None, None, :], -1e9).softmax(-1) @ v.double()
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    assert torch.equal(out[out.isinf()] > 0, want[want.isinf()] > 0)
    assert bool(out.isfinite().all()) == (kind in ("v huge", "v ramp"))
    ok = want.isfinite()
    size = v.double().abs().where(v.isfinite(), torch.zeros((), dtype=torch.float64)).amax(2, keepdim=True).clamp(min=1.0).expand_as(want)
    assert ((out.double() - want).abs()[ok] <= 2e-5 * size[ok]).all()


@pytest.mark.parametrize("generic", [False, True])
def test_output_gate_in_float32(af3, generic):
    """sigmoid of gates from 5 to 18 (times 1): half an ulp of 1 + e is 2^-24, of the quotient 2^-25, and what the exponential is off by stays
    below 0.04 * 2^-24 there.  (A reciprocal good to one ulp: 1.66 * 2^-24.)"""
    from af3_kernels_amd import ops
    gate = torch.linspace(5, 18, 4096 * 32, device="cuda").view(1, 1, 4096, 32)
    one = torch.ones_like(gate)
    out = ops._dpa_forward_impl(one, one, one, None, None, ops._DTYPE_CODE[torch.float32], generic, gate=gate)
    torch.cuda.synchronize()
    assert (out.double() - torch.sigmoid(gate.double())).abs().max() <= 1.54 * 2 ** -24


@pytest.mark.parametrize("S,N,C,head", [(1, 48, 128, 4), (1, 64, 384, 16), (1, 200, 384, 16), (5, 300, 768, 16), (1, 130, 96, 4), (1, 2048, 768, 16)])
def test_self_attention_has_the_same_bits_on_every_route(af3, S, N, C, head):
    """The first call on a set of weights, later ones, a mask that is not bool, tokens that are not contiguous or not aligned: prepared by the native host side
    or in Python, the same kernels (among the shapes: products that this library computes and one it leaves to the library GEMM)."""
    g = torch.Generator(device="cuda").manual_seed(N)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    x = r(N, C) if S == 1 else r(S, N, C)
    ws = [af3.vnni_repack_tensor(r(C, C) * C ** -0.5, 2, C // head) for _ in range(4)]
    qb, bias, mask = r(C), r(head, N, N), torch.rand(N, generator=g, device="cuda") < 0.9
    call = lambda x, mask: af3.self_attention_cpp(x, mask, bias, ws[0], qb, ws[1], ws[2], ws[3], head)
    first = call(x, mask)
    assert torch.equal(first, call(x, mask))
    assert torch.equal(first, call(x, mask.float()))
    assert torch.equal(first, call(torch.cat([x, x], -1)[..., :C], mask))
    odd = torch.empty(x.numel() + 1, device="cuda", dtype=torch.bfloat16)[1:].view(x.shape).copy_(x)   # off a 16-byte boundary
    if S * N * 4 * C * C <= 6e9 and C % 64 == 0:   # (a library GEMM may choose by the address)
        assert torch.equal(first, call(odd, mask)) and torch.equal(first, call(odd, mask.float()))


@pytest.mark.parametrize("C,head,dtype,attempts", [(128, 4, torch.float32, 1), (96, 4, torch.bfloat16, 1), (128, 4, torch.bfloat16, 2)])
def test_grid_block_asks_the_native_host_side_once(af3, monkeypatch, C, head, dtype, attempts):
    """A call that the native block does not take (here by its type, its channels, or a mask that is not bool) goes to Python after one attempt and
    derives nothing that it does not read; only the first call on a set of weights it may take asks twice."""
    from af3_kernels_amd import fused
    seen = []

    class Counting:
        def __getattr__(self, name):
            fn = getattr(host, name)
            return (lambda *a: seen.append(name) or fn(*a)) if callable(fn) else fn

    host = fused._host
    monkeypatch.setattr(fused, "_host", Counting())
    mod = af3.GridSelfAttentionCpp(C, head).to("cuda", dtype).eval().requires_grad_(False)
    pair, keep = torch.randn(40, 40, C, device="cuda").to(dtype), torch.ones(40, 40, device="cuda")
    mod(pair, keep)
    assert seen.count("grid_block") == attempts
    del seen[:]
    mod(pair, keep)
    assert seen.count("grid_block") == 1
    assert host.recalls(host.OUT_PROJ_T, mod.out_proj) == (attempts == 2)


@pytest.mark.parametrize("B,H,L,D", [(16, 2, 160, 32), (17, 2, 165, 24), (3, 2, 164, 32), (2, 1, 72, 32), (7, 3, 392, 16)])   # bias staged, from the workspace, read in place; 2 to 4 rows
@pytest.mark.parametrize("kind", ["45", "60", "68", "120", "60, large v"])
def test_shared_bias_quick_and_careful_walks(af3, oracle, B, H, L, D, kind):
    """Logits that rise far above the first tile's: row sums of 2^65 to 2^98 let the walk without sum checks stand, larger ones, results
    that overflow under the old reference (values of 2^120 at 2^86) send the workgroup through the careful walk."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g) < 0.8
    keep[:, 0] = keep[:, L - 1] = True
    rows = [1, 40, L - 1]
    bias[:, rows, L - 1] = float(kind.split(",")[0])
    if "large" in kind:
        v[B - 1, :, L - 1] *= 2.0 ** 120
    prev = af3.set_rows_kernel("always")
    try:
        print("case", B, H, L, D, kind, flush=True)
        out = f32np(af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()))
        torch.cuda.synchronize()
    finally:
        af3.set_rows_kernel(prev)
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias))
    assert np.isfinite(out).all()
    scale = np.maximum(1.0, np.abs(f32np(v)).max(axis=2, keepdims=True) * 2.0 ** -2) if "large" in kind else 1.0   # (of the column's largest value)
    assert (np.abs(out - want) / scale).max() <= 2e-2


@pytest.mark.parametrize("B,H,L,D", [(404, 4, 300, 32), (261, 4, 264, 24), (130, 8, 512, 32), (96, 8, 640, 16), (500, 4, 200, 8), (128, 2, 1281, 32)])   # 3 of 3, 2 of 4 and 2 of 2 query tiles one behind the other (the last with a gate, the second, fourth and sixth: single ones); last ones in which one to three wavefronts have rows
@pytest.mark.parametrize("kind", ["random", "no bias", "first tile", "none", "120", "120 and none"])
@pytest.mark.parametrize("gated", [False, True])
def test_shared_bias_query_tiles_in_one_workgroup(af3, B, H, L, D, kind, gated):
    """Workgroups that walk several query tiles: every row of every tile, keys that end in the first tile, workgroups that walk carefully from the
    start, single query tiles whose sums send only these through the careful walk at the end."""
    from af3_kernels_amd import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(L + D)
    q, k, v, gate = (torch.randn(B, H, L, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))
    bias = torch.randn(H, L, L, generator=g, device="cuda").to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g, device="cuda") < 0.8
    keep[:, 0] = keep[:, L - 1] = True
    if kind == "first tile":
        keep[:, 20:] = False
    if "none" in kind:
        keep[B // 2] = False
    if "120" in kind:
        bias[:, [3, L // 2, L - 2], L - 1] = 120.0   # (rows of the first, a middle and the last query tile)
    print("case", B, H, L, D, kind, gated, flush=True)
    out = ops._dpa_forward_impl(q, k, v, ops._lift_mask(keep, L), None if kind == "no bias" else bias, _lib.AF3_BF16, False, gate=gate if gated else None).float()
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    for b in range(0, B, 32):   # (float32 on the GPU, some batch rows at a time)
        qs, ks, vs = (t[b:b + 32].float().contiguous() for t in (q, k, v))
        s = torch.matmul(qs * D ** -0.5, ks.transpose(-1, -2).contiguous())
        if kind != "no bias":
            s += bias.float()
        w = torch.softmax(s.masked_fill(~keep[b:b + 32, None, None, :], -1e9), -1)
        want = torch.matmul(w, vs)
        if gated:
            want *= torch.sigmoid(gate[b:b + 32].float())
        assert (out[b:b + 32] - want).abs().max().item() <= 2e-2   # (bf16 q, k, v and probabilities; |v| < 6)


@pytest.mark.parametrize("B,H,L,D", [(3, 2, 1, 32), (2, 1, 3, 16), (4, 2, 4, 32), (3, 2, 37, 32), (2, 2, 255, 24), (3, 1, 257, 32), (2, 1, 2047, 32), (2, 1, 2049, 32), (3, 1, 2306, 16),
                                     (4, 1, 2013, 32), (3, 1, 1984, 32)])   # (the last two: around the 64 KB of LDS that a launch gets without asking)
@pytest.mark.parametrize("kind", ["random", "last", "head", "middle", "none", "bytes", "no mask"])
def test_shared_bias_mask_rows(af3, oracle, B, H, L, D, kind):
    """The shared-bias kernel's key masks: rows shorter than one load, at odd addresses, ending inside a load, longer than what is requested
    ahead; the only live keys at either end; batch rows without any; keep bytes other than 1."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L + 1, generator=g)[:, 1:] < 0.8
    if kind != "random":
        keep[1] = False
        keep[1, {"last": slice(L - 1, L), "head": slice(0, 1), "middle": slice(L // 2, L // 2 + 2)}.get(kind, slice(0, 0))] = True
    dev = keep.to(torch.uint8).mul(0x80).cuda().view(torch.bool) if kind == "bytes" else keep.cuda()
    prev = af3.set_rows_kernel("always")
    try:
        print("case", B, H, L, D, kind, flush=True)
        out = f32np(af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), None if kind == "no mask" else dev, bias.cuda()))
        torch.cuda.synchronize()
    finally:
        af3.set_rows_kernel(prev)
    if kind == "no mask":
        keep = torch.ones(B, L, dtype=torch.bool)
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias))
    assert np.abs(out - want).max() <= 2e-2   # (bf16 q, k, v and probabilities; |v| < 5)


@pytest.mark.parametrize("B,H,L,D,with_bias", [(1, 2, 1, 64, True), (1, 2, 3, 56, True), (2, 1, 4, 32, False), (1, 1, 65, 64, True), (1, 2, 255, 56, True), (5, 4, 300, 32, False), (1, 1, 1027, 64, True), (2, 2, 770, 24, False), (1, 1, 4161, 64, True), (1, 1, 8190, 64, False)])
@pytest.mark.parametrize("kind", ["random", "tail", "last", "head", "late", "gap", "none", "bytes", "no mask"])
def test_one_row_mask_rows(af3, oracle, B, H, L, D, with_bias, kind):
    """The one-row kernel's key masks: rows shorter than one load, at odd addresses, ending inside a load, of more than 64 tiles; live tiles that
    are the first of the row, or not; batch rows without any; keep bytes other than 1."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16) if with_bias else None
    keep = torch.rand(B, L + 1, generator=g)[:, 1:] < 0.8
    if kind in ("last", "head", "none"):
        keep[B - 1] = False
        keep[B - 1, {"last": slice(L - 1, L), "head": slice(0, 1), "none": slice(0, 0)}[kind]] = True
    elif kind in ("tail", "late", "gap"):
        keep[:, {"tail": slice(L - L // 3, L), "late": slice(0, L // 3), "gap": slice(L // 4, L // 2)}[kind]] = False
    dev = keep.to(torch.uint8).mul(0x80).cuda().view(torch.bool) if kind == "bytes" else keep.cuda()
    prev = af3.set_rows_kernel("never")
    try:
        print("case", B, H, L, D, kind, flush=True)
        out = f32np(af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), None if kind == "no mask" else dev, bias.cuda() if with_bias else None))
        torch.cuda.synchronize()
    finally:
        af3.set_rows_kernel(prev)
    if kind == "no mask":
        keep = torch.ones(B, L, dtype=torch.bool)
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias) if with_bias else np.zeros((H, L, L), np.float32))
    assert np.abs(out - want).max() <= 2e-2   # (bf16 q, k, v and probabilities; |v| < 5)


@pytest.mark.parametrize("B,H,L,D", [(1, 2, 1, 32), (2, 1, 3, 8), (2, 2, 4, 64), (1, 2, 31, 32), (3, 4, 255, 32), (2, 1, 1026, 20), (1, 1, 4161, 32), (70, 4, 130, 32), (1, 1, 8190, 16)])
@pytest.mark.parametrize("kind", ["random", "tail", "last", "head", "late", "gap", "none", "bytes", "no mask"])
def test_fp32_mask_rows(af3, oracle, B, H, L, D, kind):
    """The fp32 matrix kernel's key masks: rows shorter than one load, at odd addresses, ending inside a load, of more than 64 tiles; live tiles that
    are the first of the row, or not; batch rows without any; keep bytes other than 1."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g)
    keep = torch.rand(B, L + 1, generator=g)[:, 1:] < 0.8
    if kind in ("last", "head", "none"):
        keep[B - 1] = False
        keep[B - 1, {"last": slice(L - 1, L), "head": slice(0, 1), "none": slice(0, 0)}[kind]] = True
    elif kind in ("tail", "late", "gap"):
        keep[:, {"tail": slice(L - L // 3, L), "late": slice(0, L // 3), "gap": slice(L // 4, L // 2)}[kind]] = False
    dev = keep.to(torch.uint8).mul(0x80).cuda().view(torch.bool) if kind == "bytes" else keep.cuda()
    print("case", B, H, L, D, kind, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), None if kind == "no mask" else dev, bias.cuda()).cpu().numpy()
    torch.cuda.synchronize()
    if kind == "no mask":
        keep = torch.ones(B, L, dtype=torch.bool)
    want = oracle.dpa_formula(q.numpy(), k.numpy(), v.numpy(), keep.numpy(), bias.numpy())
    assert np.abs(out - want).max() <= 1e-4   # (the fp32 tier)


@pytest.mark.parametrize("B,H,L,D,whole", [(2, 4, 40, 8, 8), (1, 16, 200, 16, 16), (9, 4, 57, 32, 32), (2, 4, 512, 32, 32), (1, 5, 1155, 16, 16),
                                           (1, 16, 300, 24, 8), (1, 16, 130, 40, 24), (2, 3, 257, 48, 16)])
def test_strips_do_not_round_q(af3, oracle, B, H, L, D, whole):
    """head_dim 8 and 16 (q's second term in the padding), 32 (in instructions of its own) and the columns of 24, 40 and 48 whose second
    term the padding holds (q is zero in the others): what is rounded is each weight, once, the row sum's weights with it, and the result."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).mul(m).to(torch.bfloat16) for m in (6.0, 1.0, 1.0))
    q[..., whole:] = 0
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.ones(B, L, dtype=torch.bool)
    print("case", B, H, L, D, flush=True)
    out = f32np(af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()))
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias))
    size = oracle.dpa_formula(f32np(q), f32np(k), np.abs(f32np(v)), keep.numpy(), f32np(bias))
    # half a unit in the last of eight bits, 2^-8 at most, each: a weight, the sum of the weights, the result; q to 2^-16 (2^-8 / 8 for sums of |q k| up to 2^5)
    assert (np.abs(out - want) <= 3.125 * 2.0 ** -8 * size + 1e-6).all()
    # in rms those three are independent and each below a third of its maximum on average
    assert np.sqrt(np.mean((out - want) ** 2)) <= 2.0 ** -9 * np.sqrt(np.mean(size ** 2))


@pytest.mark.parametrize("B,H,L,D", [(2, 4, 40, 8), (1, 16, 50, 16), (1, 16, 257, 16), (37, 4, 37, 32), (2, 4, 512, 32), (3, 4, 63, 24), (1, 16, 290, 24), (1, 16, 769, 24), (1, 16, 200, 40), (1, 5, 1155, 40), (1, 16, 50, 48), (1, 16, 513, 48)])
@pytest.mark.parametrize("kind", ["k+inf", "k-inf", "k nan", "q inf", "v+inf", "v both"])
def test_strips_infinities_act_as_in_the_formula(af3, B, H, L, D, kind):
    """Infinities and NaN of live keys in each chunk of eight head columns, with and without a second term of q: NaN rows where the formula has
    them, every other row as without them."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g) < 0.8
    at = [(i % B, i % H, (L // 3 + 7 * i) % L, 8 * i + (i + 3) % 8) for i in range(D // 8)]   # (one key per chunk)
    inf = float("inf")
    for b, h, j, c in at:
        keep[b, j] = True
        if kind[0] == "k":
            k[b, h, j, c] = {"k+inf": inf, "k-inf": -inf, "k nan": float("nan")}[kind]
        elif kind == "q inf":
            q[b, h, j, c] = inf
        else:
            v[b, h, j, c] = inf
            if kind == "v both":
                keep[b, j - 1] = True
                v[b, h, j - 1, c] = -inf
    print("case", B, H, L, D, kind, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()).cpu().double()
    s = (q.double() @ k.double().transpose(-1, -2)) * D ** -0.5 + bias.double()
    want = s.masked_fill(~keep[:, None, None, :], -1e9).softmax(-1) @ v.double()
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    assert torch.equal(out[out.isinf()] > 0, want[want.isinf()] > 0)
    ok = want.isfinite()
    assert ((out - want).abs()[ok] <= 2e-2).all()   # (bf16's budget)


@pytest.mark.parametrize("B,H,L,D", [(1, 1, 32, 24), (2, 3, 33, 8), (1, 16, 50, 48), (37, 4, 37, 32), (1, 16, 257, 32), (1, 16, 290, 24), (1, 16, 513, 48), (1, 5, 1155, 16), (1, 16, 769, 24), (1, 16, 1040, 48)])
@pytest.mark.parametrize("kind", ["far", "-1e9", "-inf", "-inf, tail", "window", "misleading", "scattered"])
def test_strips_rows_masked_through_the_bias(af3, B, H, L, D, kind):
    """Query rows whose biases all lie far below zero, rows of which only the neighbourhood of the diagonal does not, and rows
    whose two samples are no sign of the rest."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g) < 0.8
    keep[:, L // 3] = True
    i = torch.arange(L)
    if kind in ("far", "-1e9") or "-inf" in kind:
        bias[:, L - L // 5:] = {"far": -3.0e4, "-1e9": -1.0e9}.get(kind, float("-inf"))
        if "tail" in kind:   # (wavefronts without a live key beside others that have some)
            keep[:, L // 3 + 1:] = False
    elif kind == "window":
        keep[:] = True
        bias[:, (i[:, None] - i[None]).abs() > 20] = -3.0e4
    elif kind == "misleading":
        bias[:, i, i] = -3.0e4
        bias[:, i, (i + L // 2) % L] = -3.0e4
        bias[:, ::2, : L // 4] = -3.0e4
    else:
        bias[:, ::5] = torch.linspace(-300.0, -180.0, L)
        bias[:, 1::7] -= 45
    print("case", B, H, L, D, kind, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()).cpu().float()
    # one batch row takes biases down to -2^126, several down to -2^16 (q.k still counts there)
    lowest = -2.0 ** 126 if B == 1 else -2.0 ** 16
    s = (q.float() @ k.float().transpose(-1, -2)) * D ** -0.5 + bias.float().clamp(min=lowest)
    rows = L - L // 5 if "-inf" in kind and B == 1 else L   # (beyond these a dropped key's logit is no lower)
    s[:, :, :rows].masked_fill_(~keep[:, None, None, :], float("-inf"))
    want = s.softmax(-1) @ v.float()
    assert (out - want).abs().max() <= 2e-2   # (bf16's budget; a logit at -3e4 or -2^16 has steps of 2^-9 or 2^-8)


@pytest.mark.parametrize("B,H,L,D", [(1, 1, 32, 24), (2, 3, 33, 8), (1, 16, 50, 48), (1, 16, 257, 32), (1, 16, 290, 24), (2, 16, 300, 48), (1, 5, 1155, 16)])
@pytest.mark.parametrize("kind", ["-inf", "+inf", "nan", "huge", "far", "q"])
def test_strips_without_a_live_key_give_the_mean(af3, B, H, L, D, kind):
    """A batch row without a live key: the mean of V over all keys, whatever its logits would have been."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    if kind == "q":   # (with finite keys)
        q[:, :, ::3, 1] = float("inf")
        q[:, :, 1::3] = 1.0e38
    elif kind == "far":   # (rows that look masked through their bias, down to some of -2^125)
        bias[:] = -float("inf")
        i = torch.arange(L)
        bias[:, i, i] = -(2.0 ** 125)
    else:
        at = torch.rand(H, L, L, generator=g) < 0.1
        bias[at] = {"-inf": -float("inf"), "+inf": float("inf"), "nan": float("nan"), "huge": 2.0 ** 100}[kind]
    keep = torch.zeros(B, L, dtype=torch.bool)
    keep[1:] = True
    print("case", B, H, L, D, kind, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()).cpu().double()
    want = v[0].double().mean(1, keepdim=True).expand(H, L, D)
    # weights of 1 are exact: fp32 sums and quotient (L 2^-24 of sums of |v| up to 5 on average), the result rounded to bf16
    assert ((out[0] - want).abs() <= 2.0 ** -8 * want.abs() + L * 2.0 ** -24 * 5).all()


@pytest.mark.parametrize("H,L,D,first", [
    (2, 7872, 48, 1), (2, 7873, 48, 0), (2, 8096, 48, 1), (2, 8097, 40, 0), (2, 8191, 48, 0), (2, 8192, 48, 1), (2, 8192, 32, 1),   # four blocks, rows at any address: the most LDS a workgroup takes
    (3, 8192, 48, 0), (2, 8192, 40, 0),                              # two workgroups per compute unit
    (9, 1953, 48, 0), (1, 3201, 24, 0), (1, 3296, 24, 1), (1, 4640, 16, 0), (1, 8191, 8, 0),   # around and above the 64 KB that a launch gets without asking
])
def test_strips_of_long_rows(af3, oracle, H, L, D, first):
    """Every length up to 8192 is served, whatever part of a compute unit's LDS its mask tables leave."""
    g = torch.Generator(device="cuda").manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(first + H * L * L, generator=g, device="cuda", dtype=torch.bfloat16)[first:].view(H, L, L)
    keep = torch.rand(L, generator=g, device="cuda") < 0.8
    keep[0] = True
    print("case", H, L, D, first, flush=True)
    out = af3.dot_product_attention_cpp(q, k, v, keep, bias)[0, :, ::13].double()
    torch.cuda.synchronize()
    s = (q[0, :, ::13].double() @ k[0].double().transpose(-1, -2).contiguous()) * D ** -0.5 + bias[:, ::13].double()
    want = s.masked_fill(~keep, -1e9).softmax(-1) @ v[0].double()
    assert (out - want).abs().max() <= 2e-2   # (bf16's budget)


@pytest.mark.parametrize("B,H,L,D", [
    (1, 1, 32, 24), (2, 3, 33, 8), (1, 16, 50, 48), (5, 4, 63, 32), (37, 4, 37, 32),   # four wavefronts, one to three blocks of 16 rows; lengths around a tile
    (1, 16, 257, 32), (1, 16, 290, 24), (1, 16, 513, 48), (1, 16, 640, 40), (1, 5, 1155, 16),   # eight
    (1, 16, 769, 24), (1, 16, 900, 24), (1, 16, 1040, 48),                                     # four blocks; two workgroups per compute unit
    (1, 2, 2050, 48),                                                                          # nine tiles per wavefront
])
@pytest.mark.parametrize("kind", ["random", "tail", "one", "none", "low", "high", "v inf"])
def test_strips(af3, oracle, B, H, L, D, kind):
    """The kernel for biases read in place: its forms at the edges of tiles and strips, masks that leave wavefronts without a live tile,
    rows whose sums leave the range of the walk without a reference."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g) < 0.8
    keep[:, 0] = True
    if kind == "tail":
        keep[:, L - L // 3:] = False
    elif kind in ("one", "none"):
        keep[:] = False
        keep[:, L // 2] = kind == "one"
    elif kind == "low":
        bias[:, ::3] -= 120
    elif kind == "high":
        bias[:, 1::3, L - 1] = 100.0
        bias[:, 2::5, : L // 2] = 90.0
        keep[:, L - 1] = True
    elif kind == "v inf":
        keep[:, L - 2] = True
        v[:, :, L - 2, D - 1] = float("inf")
    print("case", B, H, L, D, kind, flush=True)
    out = f32np(af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()))
    if kind == "v inf":   # (weights are positive, unless they round to zero)
        assert np.isposinf(out[..., D - 1]).mean() > 0.9
        out, v = out[..., : D - 1], v[..., : D - 1]
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias)) if kind != "v inf" else oracle.dpa_formula(f32np(q), f32np(k), f32np(torch.nn.functional.pad(v, (0, 1))), keep.numpy(), f32np(bias))[..., : D - 1]
    # (a bias of -120 or 100 leaves its logit steps of 2^-17 or finer; 2e-2 is bf16's budget)
    assert np.abs(out - want).max() <= 2e-2


@pytest.mark.parametrize("B,H,L,D", [(1, 16, 640, 24), (1, 16, 641, 24), (1, 16, 672, 48), (1, 16, 641, 40), (1, 8, 800, 24), (1, 8, 897, 48), (1, 8, 1185, 24),
                                     (1, 16, 255, 24), (3, 16, 257, 24), (3, 16, 289, 48)])   # 20, 21, 25, 29 and 38 tiles for eight wavefronts, 8 to 10 for four
@pytest.mark.parametrize("kind", ["random", "three tiles", "one"])
def test_strips_on_both_sides_of_the_even_walk(af3, oracle, B, H, L, D, kind):
    """The forms whose wavefronts go by age and those in which the ones behind go first, with few live tiles too."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(B, L, generator=g) < 0.8
    keep[:, 0] = True
    if kind != "random":
        keep[:, 96 if kind == "three tiles" else 1:] = False
    prev = af3.set_rows_kernel("never")
    try:
        print("case", B, H, L, D, kind, flush=True)
        out = f32np(af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), bias.cuda()))
    finally:
        af3.set_rows_kernel(prev)
    assert np.abs(out - oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias))).max() <= 2e-2   # (bf16's budget)


@pytest.mark.parametrize("B,H,L", [(5, 2, 72), (3, 2, 133), (404, 4, 300), (130, 8, 512)])   # single query tiles; several to a workgroup
@pytest.mark.parametrize("D", [8, 16, 24, 32])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("out_type", [torch.bfloat16, torch.float32])
def test_shared_bias_stores_head_dim_columns(af3, B, H, L, D, gated, out_type):
    """Every column of every row, and nothing beside them: rows of the result that lie apart keep what stands between them."""
    from af3_kernels_amd import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(L + D)
    q, k, v, gate = (torch.randn(B, H, L, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))
    bias = torch.randn(H, L, (L + 7) // 8 * 8, generator=g, device="cuda").to(torch.bfloat16)[..., :L]
    room = torch.full((B, L + 1, H, D + 8), 7.0, dtype=out_type, device="cuda")
    prev = af3.set_rows_kernel("always")
    try:
        print("case", B, H, L, D, gated, out_type, flush=True)
        ops._dpa_forward_impl(q, k, v, None, bias, _lib.AF3_BF16, False, gate=gate if gated else None, out=room[:, :L, :, :D].transpose(1, 2))
        torch.cuda.synchronize()
    finally:
        af3.set_rows_kernel(prev)
    assert (room[:, L] == 7).all() and (room[..., D:] == 7).all()
    out = room[:, :L, :, :D].transpose(1, 2)
    for b in range(0, B, 32):   # (float32 on the GPU, some batch rows at a time)
        qs, ks, vs = (t[b:b + 32].float().contiguous() for t in (q, k, v))
        want = torch.matmul(torch.softmax(torch.matmul(qs * D ** -0.5, ks.transpose(-1, -2).contiguous()) + bias.float(), -1), vs)
        if gated:
            want *= torch.sigmoid(gate[b:b + 32].float())
        assert (out[b:b + 32].float() - want).abs().max().item() <= 2e-2   # (bf16 q, k, v and probabilities; |v| < 6)


def _rows_plan(q, k, v, out, bias, gate):
    """The shared-bias kernel's launches of a call: (batch rows per wavefront, bias mode, query tiles per workgroup)."""
    import ctypes
    from af3_kernels_amd import _lib, ops
    p = ops._fill_params(q, k, v, None, bias, out, _lib.AF3_BF16, False, gate=gate)
    p.workspace, p.workspace_bytes = 1 << 40, 1 << 40   # (nothing follows the address)
    plan = (ctypes.c_int64 * 6 * 3)()
    n = _lib.load().af3_dpa_rows_plan(ctypes.byref(p), plan)
    return [(launch[0], launch[1], launch[3]) for launch in plan[:n]]


@pytest.mark.parametrize("B,H,L,D,gated,want", [
    (460, 4, 460, 32, False, (4, 1, 4)), (404, 4, 300, 32, False, (2, 1, 3)), (404, 4, 300, 32, True, (2, 1, 3)),   # two to four batch rows per wavefront, as many tiles
    (400, 4, 400, 32, False, (2, 3, 2)), (400, 4, 400, 32, True, (2, 3, 2)),
    (384, 4, 384, 32, False, (3, 3, 3)), (384, 4, 384, 32, True, (3, 3, 3)),
    (768, 2, 768, 32, False, (3, 1, 2)), (768, 2, 768, 32, True, (3, 1, 2)),
    (461, 4, 300, 32, False, (4, 1, 3)), (640, 2, 768, 32, False, (4, 1, 2)),
    (128, 16, 512, 32, False, (4, 3, 2)), (128, 8, 768, 32, False, (4, 3, 3)), (160, 4, 640, 32, False, (4, 3, 2)),
])
@pytest.mark.parametrize("layout", ["dense", "per head"])   # [B, H, L, D] each; k, v, q and gate side by side for each token and head, the result [B, L, H, D]
@pytest.mark.parametrize("kind", ["random", "no bias", "first tile", "none", "120", "k inf"])
def test_shared_bias_forms_of_the_longer_walk(af3, B, H, L, D, gated, want, layout, kind):
    """Every number of batch rows per wavefront, place of the bias and number of query tiles one behind the other that a call can meet: keys that end
    in the first tile, a batch row without a live key (walks carefully from the start), query tiles walked again, an infinity in K."""
    from af3_kernels_amd import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(L + D)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    if layout == "dense":
        k, v, q, gate = (r(B, H, L, D) for _ in range(4))
        out = torch.empty_like(q)
    else:
        k, v, q, gate = r(B, L, H, 4, D).permute(3, 0, 2, 1, 4).unbind(0)
        out = torch.empty(B, L, H, D, device="cuda", dtype=torch.bfloat16).transpose(1, 2)
    gate = gate if gated else None
    bias = None if kind == "no bias" else r(H, L, L)
    keep = torch.rand(B, L, generator=g, device="cuda") < 0.8
    keep[:, 0] = keep[:, 70] = keep[:, L - 1] = True
    if kind == "first tile":
        keep[:, 20:] = False
    elif kind == "none":
        keep[B // 2] = False
    elif kind == "120":
        bias[:, [3, L // 2, L - 2], L - 1] = 120.0   # (rows of the first, a middle and the last query tile)
    elif kind == "k inf":
        k[B // 2, 1, 70, 1] = float("inf")
    plan = _rows_plan(q, k, v, out, bias, gate)
    assert plan[0][::2] == want[::2] and plan[0][1] == (0 if bias is None else want[1])
    print("case", B, H, L, D, gated, layout, kind, flush=True)
    ops._dpa_forward_impl(q, k, v, ops._lift_mask(keep, L), bias, _lib.AF3_BF16, False, gate=gate, out=out)
    torch.cuda.synchronize()
    for b in range(0, B, 32):   # (float32 on the GPU, some batch rows at a time)
        qs, ks, vs = (t[b:b + 32].float().contiguous() for t in (q, k, v))
        s = torch.matmul(qs * D ** -0.5, ks.transpose(-1, -2).contiguous())
        if bias is not None:
            s += bias.float()
        ref = torch.matmul(torch.softmax(s.masked_fill(~keep[b:b + 32, None, None, :], -1e9), -1), vs)
        if gated:
            ref *= torch.sigmoid(gate[b:b + 32].float())
        got, nan = out[b:b + 32].float(), ref.isnan()
        if kind == "k inf" and b <= B // 2 < b + 32:   # (this kernel's NaN rows take the query row 16 further on or back with them, never another head or batch row)
            block = slice(B // 2 - b, B // 2 - b + 1), slice(1, 2)
            assert nan[block].any() and (got[block].isnan() >= nan[block]).all()
            nan[block] |= got[block].isnan()
        assert torch.equal(got.isnan(), nan)
        assert (got - ref).masked_fill(nan, 0.0).abs().max().item() <= 2e-2   # (bf16 q, k, v and probabilities; |v| < 6)


@pytest.mark.parametrize("row,taken", [((1 << 24) - 8, True), (1 << 24, False)])
@pytest.mark.parametrize("which", ["q", "out"])
def test_shared_bias_row_strides(af3, which, row, taken):
    """Rows of q or of the result that lie up to 2^24 elements apart are addressed by the shared-bias kernel; calls with rows further apart go to the
    one-row kernel."""
    from af3_kernels_amd import _lib, ops
    B, H, L, D = 2, 1, 133, 32
    g = torch.Generator(device="cuda").manual_seed(row)
    q, k, v = (torch.randn(B, H, L, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    bias = torch.randn(H, L, 136, generator=g, device="cuda").to(torch.bfloat16)[..., :L]
    wide = torch.empty((L - 1) * row + B * D, device="cuda", dtype=torch.bfloat16).as_strided((B, H, L, D), (D, D, row, 1))
    out = torch.empty_like(q)
    if which == "q":
        qs, outs = wide.copy_(q), out
    else:
        qs, outs = q, wide
    prev = af3.set_rows_kernel("always")
    try:
        assert bool(_rows_plan(qs, k, v, outs, bias, None)) == taken
        print("case", which, row, flush=True)
        ops._dpa_forward_impl(qs, k, v, None, bias, _lib.AF3_BF16, False, out=outs)
        torch.cuda.synchronize()
    finally:
        af3.set_rows_kernel(prev)
    want = torch.matmul(torch.softmax(torch.matmul(q.float() * D ** -0.5, k.float().transpose(-1, -2).contiguous()) + bias.float(), -1), v.float())
    assert (outs.float() - want).abs().max().item() <= 2e-2   # (bf16 q, k, v and probabilities; |v| < 6)
