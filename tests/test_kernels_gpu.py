"""Each kernel alone against a plain reference, at other sizes than the engine's tiny models
use: sizes that are no power of two, head sizes in steps of 16, grouped heads, windows, pages
scattered over the pool, and a pool that is NaN wherever nothing was written."""
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import helpers
import plain_gpt2 as P

pytestmark = pytest.mark.gpu
DEV = helpers.DEVICE


@pytest.fixture(scope="module")
def ops():
    from deliverance_amd.kernels import ops as o
    return o


def bf(x):
    return x.to(torch.bfloat16)


# ----------------------------------------------------------------------------- embedding, norm
@pytest.mark.simt_quick
@pytest.mark.parametrize("table_dtype", [torch.float32, torch.bfloat16])
def test_embed(ops, table_dtype):
    g = torch.Generator().manual_seed(0)
    V, Pn, E, N = 1000, 77, 200, 37
    wte = torch.randn(V, E, generator=g).to(table_dtype).to(DEV)
    wpe = torch.randn(Pn, E, generator=g).to(table_dtype).to(DEV)
    tok = torch.randint(0, V, (N,), generator=g, dtype=torch.int32).to(DEV)
    pos = torch.randint(0, Pn, (N,), generator=g, dtype=torch.int32).to(DEV)
    out = torch.empty(N, E, device=DEV)
    ops.embed(tok, pos, wte, wpe, out)
    want = wte.float()[tok.long()] + wpe.float()[pos.long()]
    assert torch.equal(out, want)
    ops.embed(tok, pos, wte, None, out)
    assert torch.equal(out, wte.float()[tok.long()])


@pytest.mark.simt_quick
def test_embed_scale_and_row_copies(ops):
    g = torch.Generator().manual_seed(2)
    V, Pn, E, N = 300, 50, 72, 21
    wte, wpe = bf(torch.randn(V, E, generator=g)).to(DEV), bf(torch.randn(Pn, E, generator=g)).to(DEV)
    tok = torch.randint(0, V, (N,), generator=g, dtype=torch.int32).to(DEV)
    pos = torch.randint(0, Pn, (N,), generator=g, dtype=torch.int32).to(DEV)
    out = torch.empty(N, E, device=DEV)
    ops.embed(tok, pos, wte, wpe, out, scale=8.5)
    assert torch.equal(out, wte.float()[tok.long()] * 8.5 + wpe.float()[pos.long()])
    # rows gathered and converted; rows added into the 32-bit stream
    rows = torch.tensor([20, 0, 7, 7, 3], dtype=torch.int32, device=DEV)
    for dt in (torch.float32, torch.bfloat16):
        dst = torch.empty(5, E, device=DEV, dtype=dt)
        ops.copy_rows(out, dst, rows=rows)
        assert torch.equal(dst, out[rows.long()].to(dt))
        dst = torch.empty(N, E, device=DEV, dtype=dt)
        ops.copy_rows(out, dst)
        assert torch.equal(dst, out.to(dt))
    acc = torch.randn(N, E, generator=g).to(DEV)
    want = acc + bf(out).float()
    ops.copy_rows(bf(out), acc, accumulate=True)
    assert torch.equal(acc, want)
    with pytest.raises(ops.KernelError, match="float32 destination"):
        ops.copy_rows(out, bf(out), accumulate=True)


@pytest.mark.simt_quick
@pytest.mark.parametrize("E,eps", [(7, 1e-5), (200, 1e-6), (1600, 1e-5), (64, 1e-1)])
def test_layernorm(ops, E, eps):
    g = torch.Generator().manual_seed(1)
    N = 19
    x = (torch.randn(N, E, generator=g) * 3 + 5).to(DEV)       # a large mean: E[x^2]-mean^2 would lose digits
    w, b = torch.randn(E, generator=g).to(DEV), torch.randn(E, generator=g).to(DEV)
    out = torch.empty(N, E, device=DEV)
    ops.layernorm(x, w, b, eps, out)
    want = F.layer_norm(x.double(), (E,), w.double(), b.double(), eps)
    assert (out.double() - want).abs().max() < 2e-5
    # bfloat16 parameters and output, gathered rows
    rows = torch.tensor([5, 0, 18, 5], dtype=torch.int32, device=DEV)
    o2 = torch.empty(4, E, device=DEV, dtype=torch.bfloat16)
    ops.layernorm(x, bf(w), bf(b), eps, o2, rows)
    want2 = F.layer_norm(x.double(), (E,), bf(w).double(), bf(b).double(), eps)[rows.long()]
    assert (o2.double() - want2).abs().max() < 4e-2
    assert torch.equal(o2[0], o2[3])
    if E == 7:   # the reference's own vector (LayerNormTest.java:40,51,77,88)
        xv = torch.tensor([[-1.1151, 0.1490, -1.0923, -1.4551, 1.3358, 0.3075, 0.6278]], device=DEV)
        o3 = torch.empty(1, 7, device=DEV)
        ops.layernorm(xv, torch.ones(7, device=DEV), torch.zeros(7, device=DEV), 1e-5, o3)
        want3 = torch.tensor([-0.9635, 0.3355, -0.9401, -1.3129, 1.5551, 0.4984, 0.8275], device=DEV)
        assert (o3[0] - want3).abs().max() < 1e-4


@pytest.mark.parametrize("E", [helpers.quick(132), helpers.quick(256), 260, helpers.quick(512), 516, 768, 1000, 1024])
def test_norms_of_many_rows(ops, E):
    """Rows of up to 1,024 columns take one wavefront or four by their number: the same bits either way, at the lines between
    the two and beside them."""
    R = 2049 if E <= 512 else 4097
    helpers.skip_in_simulation_if(E > 512)
    g = torch.Generator().manual_seed(E)
    x, src = ((torch.randn(R, E, generator=g) * 3 + 5).to(DEV) for _ in range(2))
    w, b = (torch.randn(E, generator=g).to(DEV) for _ in range(2))
    for y, dt in ((torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)):
        def norms(lo, hi):
            n, outs = hi - lo, []
            outs.append(ops.layernorm(x[lo:hi], w.to(dt), b.to(dt), 1e-5, torch.empty(n, E, dtype=y, device=DEV)))
            outs.append(ops.rmsnorm(x[lo:hi], w.to(dt), 1.0, 1e-5, torch.empty(n, E, dtype=y, device=DEV)))
            stream, h = x[lo:hi].clone(), torch.empty(n, E, dtype=y, device=DEV)
            ops.rmsnorm_add(src[lo:hi], w.to(dt), stream, 1.0, 1e-5, b.to(dt), h)
            return outs + [stream, h]
        few = norms(0, 5)
        for n in (R,) if helpers.SIMT else (511, 513, 767, 768, 1023, 1024, 2047, 2048, R - 1, R):
            many = norms(0, n)
            assert all(torch.equal(f, m[:5]) for f, m in zip(few, many)), n
            if n == R:
                assert all(torch.equal(f, m[-5:]) for f, m in zip(norms(n - 5, n), many))
        wd, bd, xd = w.to(dt).double(), b.to(dt).double(), x.double()
        rms = lambda v, gain: v / (v.square().mean(1, keepdim=True) + 1e-5).sqrt() * (1.0 + gain)
        new = xd + rms(src.double(), wd)
        for got, want in zip(many, (F.layer_norm(xd, (E,), wd, bd, 1e-5), rms(xd, wd), new, rms(new, bd))):
            tol = 2e-5 if got.dtype == torch.float32 else 2.0 ** -8       # (32-bit: as for LayerNorm above; bfloat16: one rounding)
            assert ((got.double() - want).abs() / want.abs().clamp(min=1.0)).max() < tol


# ----------------------------------------------------------------------------- products
def _gemm_case(ops, fn, M, N, K, dtype, act, accumulate, bias, out_dtype, g):
    a = (torch.randn(M, K, generator=g) * 0.5).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=g) * 0.2).to(dtype).to(DEV)
    b = torch.randn(N, generator=g).to(dtype).to(DEV) if bias else None
    base = torch.randn(M, N, generator=g).to(DEV)
    out = base.clone() if accumulate else torch.empty(M, N, device=DEV, dtype=out_dtype)
    fn(a, w, b, out, act, accumulate)
    ref = a.double() @ w.double().t()
    if bias:
        ref = ref + b.double()
    if act == "gelu_new":
        ref = F.gelu(ref, approximate="tanh")
    elif act == "gelu":
        ref = F.gelu(ref)
    elif act == "relu":
        ref = F.relu(ref)
    elif act == "silu":
        ref = F.silu(ref)
    if accumulate:
        ref = ref + base.double()
    return out.double(), ref


@pytest.mark.simt_quick
@pytest.mark.parametrize("M,N,K", [(1, 50, 24), (5, 1000, 96), (70, 200, 96), (130, 77, 200), (64, 64, 64)])
def test_gemm_plain_32bit(ops, M, N, K):
    g = torch.Generator().manual_seed(M * 1000 + N)
    for act, acc, bias in ((None, False, True), ("gelu_new", False, True), ("gelu", False, False),
                           (None, True, True), ("silu", False, True), ("relu", False, True)):
        out, ref = _gemm_case(ops, ops.linear_ref, M, N, K, torch.float32, act, acc, bias, torch.float32, g)
        assert (out - ref).abs().max() < 2e-5 * max(1.0, ref.abs().max().item())


@pytest.mark.parametrize("form", ["auto", "rows", "64x64", "32x32"])
@pytest.mark.parametrize("M,N,K", [(1, 50, 24), helpers.quick(5, 1000, 96), (16, 64, 128), helpers.quick(17, 33, 132), (65, 200, 772),
                                   (130, 77, 200), (300, 1100, 640), (16, 2100, 3072)])
def test_gemm_32bit_on_the_matrix_cores(ops, M, N, K, form):
    """Every kernel form behind ``linear_f32``: K below a group, below a chunk, cut and whole chunks; edges in M and N; a
    row has the same bits in every form and beside any other rows.  Bound: a sum in chunks of 128 loses at most
    (128 + K / 128) roundings of 2^-24 of the sum of magnitudes, which is below sqrt(K) times the operands' scale here."""
    helpers.skip_in_simulation_if(M * N * K > 4e6)
    g = torch.Generator().manual_seed(M * 1000 + N)
    fn = lambda a, w, b, out, act, acc: ops.linear_f32(a, w, b, out, act, acc, form=form)
    for act, acc, bias in ((None, False, True), ("gelu_new", False, True), (None, True, True), ("silu", False, False)):
        out, ref = _gemm_case(ops, fn, M, N, K, torch.float32, act, acc, bias, torch.float32, g)
        assert (out - ref).abs().max() < 2e-5 * max(1.0, ref.abs().max().item())
    a = (torch.randn(M, K, generator=g)).to(DEV)
    w = (torch.randn(N, K, generator=g)).to(DEV)
    o1, o2, o3 = (torch.empty(M, N, device=DEV) for _ in range(3))
    ops.linear_f32(a, w, None, o1, form=form)
    ops.linear_f32(a, w, None, o2, form="64x64" if form == "32x32" else "32x32")
    ops.linear_f32(a[M // 2:M // 2 + 1], w, None, o3[:1])
    assert torch.equal(o1, o2) and torch.equal(o1[M // 2], o3[0])


@pytest.mark.parametrize("M,N,K", [(3, 40, 4100), helpers.quick(1, 20, 6400), (2, 2100, 6400), (16, 70, 3076), (8, 24, 6404), helpers.quick(1, 9, 6404)])
def test_gemm_32bit_of_few_rows_and_many_columns_of_a(ops, M, N, K):
    """The kernel for few rows with its largest room for partial sums (K from 3,073 to 6,400), and above that the tiles; the
    same bits as the tiles.  Bound as above."""
    g = torch.Generator().manual_seed(K + N)
    for act, acc, bias in ((None, True, True), ("gelu_new", False, True)):
        out, ref = _gemm_case(ops, ops.linear_f32, M, N, K, torch.float32, act, acc, bias, torch.float32, g)
        assert (out - ref).abs().max() < 2e-5 * max(1.0, ref.abs().max().item())
    a, w = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV)
    tiles = ops.linear_f32(a, w, None, torch.empty(M, N, device=DEV), form="32x32")
    for form in ("auto", "rows", "64x64") if K <= 6400 else ("auto", "64x64"):
        assert torch.equal(ops.linear_f32(a, w, None, torch.empty(M, N, device=DEV), form=form), tiles), form


@pytest.mark.parametrize("M,N,K,bf16", [(17, 1056, 4096, True), (9, 1028, 4160, True), (16, 1600, 6400, True), (33, 2048, 4096, False),
                                        (64, 1600, 6400, True), (48, 1100, 4608, False), helpers.quick(65, 68, 2048, True), (66, 260, 2112, True), (129, 768, 3072, False),
                                        (552, 1024, 4096, True), (1025, 1024, 2112, True), (640, 2048, 6400, True)])
def test_products_shared_out_over_k(ops, M, N, K, bf16):
    """The shares' sums, added to a stream with a bias, and the norm of the new rows, whole and of repeated rows; ragged last
    shares, edges of tiles, both forms.  The bound: a running sum of K products of random sign is about sqrt(K) of them, and K roundings of 2^-24 of it add up
    like sqrt(K) of them: K products' magnitudes by 2^-24, that is 2^-24 of the sum of magnitudes; four times that."""
    helpers.skip_in_simulation_if(M * N * K > 1e7)
    n = ops.product_shares(M, N, K)
    assert n > 1
    g = torch.Generator().manual_seed(M + K)
    dt = torch.bfloat16 if bf16 else torch.float32
    a, w = bf(torch.randn(M, K, generator=g)).to(DEV), bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    bias, gain, add = (torch.randn(N, generator=g).to(dt).to(DEV) for _ in range(3))
    x = torch.randn(M, N, generator=g).to(DEV)
    partial = ops.linear_shares(a, w, torch.full((n * M, N), float("nan"), device=DEV))
    new = x.double() + a.double() @ w.double().t() + add.double()
    tol = 2.0 ** -22 * (a.float().abs() @ w.float().abs().t()).max().item()
    joined = ops.join_rows(x.clone(), partial, add)
    assert (joined.double() - new).abs().max() < tol
    kept, h = x.clone(), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.layernorm_join(kept, partial, add, gain, bias, 1e-5, h)
    assert torch.equal(kept, joined) and torch.equal(h, ops.layernorm(joined, gain, bias, 1e-5, torch.empty_like(h)))
    rows = torch.tensor([M - 1, 0, M - 1, M // 2], dtype=torch.int32, device=DEV)
    few = ops.layernorm_join(x, partial, None, gain, bias, 1e-5, torch.empty(4, N, dtype=torch.bfloat16, device=DEV), rows)
    plain = ops.join_rows(x.clone(), partial, None)
    assert torch.equal(few, ops.layernorm(plain, gain, bias, 1e-5, torch.empty_like(few), rows))


def test_products_that_are_not_shared_out_are_refused(ops):
    for M, N, K in ((8, 1600, 6400), (64, 768, 3072), (64, 1024, 4096), (100, 1024, 1024), (100, 2304, 4096), (100, 1022, 4096), (1500, 1024, 4096), (4096, 1600, 6400)):
        assert ops.product_shares(M, N, K) == 1
    a, w = (torch.zeros(s, 1024, dtype=torch.bfloat16, device=DEV) for s in (100, 1024))
    with pytest.raises(ops.KernelError):
        ops.linear_shares(a, w, torch.zeros(100, 1024, device=DEV))


def test_which_products_a_step_shares_out(ops):
    """The rule's lines; never more shares than the product can be cut into."""
    for M, N, K in ((48, 1600, 6400), (33, 1600, 6400), (64, 1280, 5120), (552, 1024, 4096), (840, 768, 3072), (1100, 1024, 4096), (1024, 1280, 5120), (66, 260, 2112), (552, 2048, 4096)):
        assert ops.step_shares(M, N, K) == ops.product_shares(M, N, K) > 1, (M, N, K)
    for M, N, K in ((32, 1600, 6400), (48, 1280, 5120), (64, 2048, 4096), (841, 768, 3072), (1300, 512, 2048), (1024, 1024, 4096), (552, 1024, 2048), (400, 2048, 4096)):
        assert ops.step_shares(M, N, K) == 1 < ops.product_shares(M, N, K), (M, N, K)
    assert ops.step_shares(64, 1024, 4096) == ops.step_shares(8, 1600, 6400) == ops.step_shares(1500, 1024, 4096) == 1


@pytest.mark.parametrize("M,N,K", [helpers.quick(3, 700, 772), helpers.quick(4, 1030, 132), (2, 250, 6400), (4, 2100, 1284), (1, 13000, 260),
                                   helpers.quick(8, 1100, 388), (5, 2050, 644), (7, 10500, 132), (8, 5000, 3072), (8, 10500, 3076),
                                   helpers.quick(9, 300, 260), (16, 1000, 6400), (33, 3000, 388), (12, 4100, 516), (16, 10240, 1028),
                                   (13, 4200, 3076), helpers.quick(4, 520, 64)])
def test_gemm_32bit_of_few_rows_by_columns(ops, M, N, K):
    """The kernel for few rows with 1 to 16 columns a workgroup, four, two and one chunk a product, few and many workgroups, K cut
    in every place of a set of chunks, and fragments straight from memory: the bits of the tiles.  Bound as above."""
    helpers.skip_in_simulation_if(M * N * K > 4e6)
    g = torch.Generator().manual_seed(M + N + K)
    out, ref = _gemm_case(ops, ops.linear_f32, M, N, K, torch.float32, None, True, True, torch.float32, g)
    assert (out - ref).abs().max() < 2e-5 * max(1.0, ref.abs().max().item())
    a, w = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV)
    rows = ops.linear_f32(a, w, None, torch.empty(M, N, device=DEV), form="rows")
    assert torch.equal(rows, ops.linear_f32(a, w, None, torch.empty(M, N, device=DEV), form="32x32"))


@pytest.mark.parametrize("M,N,K", [helpers.quick(1, 68, 64), helpers.quick(4, 1030, 132), (5, 1400, 388), helpers.quick(17, 260, 516), (8, 9300, 260), (20, 2100, 1284),
                                   (33, 1100, 1156), (48, 1024, 772), (100, 260, 3076), (3, 2500, 6400), (12, 4100, 644)])
def test_gemm_32bit_of_few_rows_both_kernels(ops, M, N, K):
    """The direct and the staged kernel, 4 to 16 columns a workgroup and K in every set of wavefronts: the bits of the tiles."""
    helpers.skip_in_simulation_if(M * N * K > 1e7)
    g = torch.Generator().manual_seed(M + N + K)
    a, w, b, x = (torch.randn(*s, generator=g).to(DEV) for s in ((M, K), (N, K), (N,), (M, N)))
    tiles = ops.linear_f32(a, w, b, x.clone(), act="gelu_new", accumulate=True, form="32x32")
    for form in ("rows_direct", "rows_staged"):
        assert torch.equal(ops.linear_f32(a, w, b, x.clone(), act="gelu_new", accumulate=True, form=form), tiles), form
    with pytest.raises(ops.KernelError):
        ops.linear_f32(torch.zeros(2, 6404, device=DEV), torch.zeros(4, 6404, device=DEV), None, torch.empty(2, 4, device=DEV), form="rows_direct")


def test_which_kernel_32bit_products_of_few_rows_take(ops):
    """The rule's lines, and never a second round of workgroups of the staged kernel for less than 16 columns each."""
    choice = ops._lib().da_gemm_f32_rows_choice
    for M, N, K in ((4, 512, 256), (8, 50257, 384), (8, 9216, 512), (4, 6144, 768), (16, 6144, 1152), (4, 3072, 1600), (12, 4100, 2048), (17, 2304, 3072), (33, 2048, 1152),
                    (8, 16384, 1024), (4, 8192, 4096)):
        assert choice(M, N, K) == 0, (M, N, K)
    for M, N, K, cols in ((4, 768, 768, 3), (4, 3072, 768, 12), (4, 50257, 768, 16), (8, 1024, 4096, 4), (16, 4800, 5120, 16), (48, 1024, 1600, 13), (100, 256, 768, 8), (1, 64, 512, 1)):
        assert choice(M, N, K) == cols, (M, N, K)
    for M in (1, 4, 5, 8, 9, 16, 17, 33, 48, 64, 100, 256):
        for N in (1, 64, 250, 256, 770, 1024, 2304, 4096, 50257):
            cols = choice(M, N, 6400)
            if 0 < cols < 16:
                assert -(-N // cols) * -(-M // (4 if M <= 4 else 8 if M <= 8 else 16)) <= 256, (M, N)


def test_gemm_32bit_writes_keys_and_values(ops):
    g = torch.Generator().manual_seed(7)
    Hq, Hkv, D, page, K = 5, 3, 20, 16, 132
    N = (Hq + 2 * Hkv) * D
    for M in (3, 70):
        n_pages = (M + page - 1) // page + 2
        a, w, bias = (torch.randn(*s, generator=g).to(DEV) for s in ((M, K), (N, K), (N,)))
        slots = torch.randperm(n_pages * page, generator=g)[:M].to(torch.int32)
        slots[M // 2] = -1
        slots = slots.to(DEV)
        c1 = torch.zeros(n_pages, 2, Hkv, page, D, device=DEV)
        c2 = torch.zeros_like(c1)
        out = torch.empty(M, N, device=DEV)
        ops.linear_f32(a, w, bias, out, kv_cache=c1, slot_map=slots, q_cols=Hq * D)
        ops.kv_write(out, Hq * D, (Hq + Hkv) * D, c2, slots, Hkv, D)
        assert torch.equal(c1, c2) and c1.abs().sum() > 0


@pytest.mark.parametrize("K", [helpers.quick(128), 132, 640, 768, 772, 1000, 1024])
@pytest.mark.parametrize("M,N", [helpers.quick(1, 300), (4, 192), (3, 1500), (4, 2304), (8, 2304), (5, 1056), (2, 4096), (8, 3075)])
def test_layer_norm_and_product_32bit_in_one_kernel(ops, M, N, K):
    """The bits of the norm's kernel and the product's, at every width of a workgroup, k that cuts a chunk and wavefronts without one; with
    and without the norm's bias, a bias and an activation, and the cache write where N is q | k | v."""
    helpers.skip_in_simulation_if(M * N * K > 300_000)
    g = torch.Generator().manual_seed(N + K)
    x = (torch.randn(M, K, generator=g) * 3 + 1).to(DEV)
    gain, add = (torch.randn(K, generator=g) + 1).to(DEV), torch.randn(K, generator=g).to(DEV)
    w, bias = torch.randn(N, K, generator=g).to(DEV), torch.randn(N, generator=g).to(DEV)
    assert ops.can_fuse_ln_f32(M, x, gain, add, w)
    D, page = 16, 16
    heads = N // (3 * D)
    cached = N % (3 * D) == 0
    slots = torch.tensor([5, -1, 16, 31, 0, 33, 47, 20][:M], dtype=torch.int32, device=DEV)
    for b, act, lb in ((bias, "gelu_new", add), (None, None, None)):
        kv = [dict(kv_cache=torch.zeros(3, 2, heads, page, D, device=DEV), slot_map=slots, q_cols=heads * D) if cached else {} for _ in range(2)]
        normed = ops.layernorm(x, gain, lb, 1e-5, torch.empty(M, K, device=DEV), None)
        two = ops.linear_f32(normed, w, b, torch.full((M, N), 7.0, device=DEV), act, **kv[0])
        one = ops.linear_ln_f32(x, gain, lb, 1e-5, w, b, torch.full((M, N), 8.0, device=DEV), act, **kv[1])
        assert torch.equal(one, two)
        if cached:
            assert torch.equal(kv[0]["kv_cache"], kv[1]["kv_cache"])
    xd = x.double()
    c = xd - xd.mean(1, keepdim=True)
    want = (c / torch.sqrt((c * c).mean(1, keepdim=True) + 1e-5) * gain.double()) @ w.double().t()
    # (sqrt(K) roundings of 6e-8 of numbers of order one, K of them: far below this)
    assert float((one.double() - want).norm() / want.norm()) < 2e-6


def test_which_steps_32bit_norm_and_product_take(ops):
    x = torch.zeros(9, 1028, device=DEV)
    gain = torch.zeros(1028, device=DEV)
    takes = lambda M, N, K: ops.can_fuse_ln_f32(M, x[:M, :K].contiguous(), gain[:K], None, torch.zeros(N, K, device=DEV))
    assert takes(4, 1, 128) and takes(1, 1025, 4) and takes(8, 1025, 128) and takes(8, 4096, 896) and takes(8, 3600, 1024)
    assert not takes(9, 2304, 768) and not takes(4, 4097, 768) and not takes(4, 2304, 1028) and not takes(4, 1024, 124)
    assert not takes(5, 1024, 768) and not takes(8, 3601, 900) and not takes(5, 2000, 124)
    w = torch.zeros(8, 256, device=DEV)
    assert not ops.can_fuse_ln_f32(1, x[:1, :256].contiguous(), gain[1:257], None, w)          # a gain that is not aligned
    with pytest.raises(ops.KernelError):
        ops.linear_ln_f32(torch.zeros(9, 256, device=DEV), gain[:256], None, 1e-5, w, None, torch.empty(9, 8, device=DEV))


@pytest.mark.simt_quick
@pytest.mark.parametrize("extra,accumulate", [(0, False), (0, True), (12, False), (12, True)])
def test_product_32bit_keeps_keys_and_values_of_any_call(ops, extra, accumulate):
    """``linear`` with a cache: columns behind q | k | v, and sums that are added to what was there; the cache holds what
    the rows hold afterwards."""
    g = torch.Generator().manual_seed(11)
    Hq, Hkv, D, page, K, M = 2, 1, 16, 16, 64, 5
    N = (Hq + 2 * Hkv) * D + extra
    a, w = (torch.randn(*s, generator=g).to(DEV) for s in ((M, K), (N, K)))
    base = torch.randn(M, N, generator=g).to(DEV)
    out = base.clone()
    slots = torch.tensor([20, 3, -1, 31, 0], dtype=torch.int32, device=DEV)
    c1, c2 = (torch.zeros(2, 2, Hkv, page, D, device=DEV) for _ in range(2))
    ops.linear(a, w, None, out, accumulate=accumulate, kv_cache=c1, slot_map=slots, q_cols=Hq * D)
    ref = a.double() @ w.double().t() + (base.double() if accumulate else 0.0)
    assert (out.double() - ref).abs().max() < 2e-5 * max(1.0, ref.abs().max().item())
    ops.kv_write(out, Hq * D, (Hq + Hkv) * D, c2, slots, Hkv, D)
    assert torch.equal(c1, c2) and bool(c1.any())


@pytest.mark.parametrize("M", [1, helpers.quick(3, mark="simt_a"), 5, 8, 12, 16, helpers.quick(17, mark="simt_a"), 40, 64,
                               helpers.quick(65, mark="simt_a"), 128, helpers.quick(200, mark="simt_a"), 513, 1100, 2048])
@pytest.mark.parametrize("N,K", [helpers.quick(96, 200, mark="simt_b"), helpers.quick(1000, 96, mark="simt_b"), (2304, 768),
                                 helpers.quick(50, 24, mark="simt_b"), helpers.quick(300, 2056, mark="simt_b"), (1030, 1160),
                                 (4200, 200), helpers.quick(4096, 8, mark="simt_b")])
def test_gemm_matrix_cores(ops, M, N, K):
    """Every kernel form behind ``linear_mfma`` (up to 4 rows and 2,048 columns: 16x16x32 products of four pieces of k, 4 or 8
    wavefronts; up to 64 rows: 16x16x32 products fed through LDS, 1 to 4 row tiles, 8 or 12 wavefronts;
    else block tiles of 64x64, 128x64 and 128x128, chosen by the number of tiles: 1,100 and 2,048 rows
    reach the larger ones), each with a last step that K cuts or a K below one slab."""
    helpers.skip_in_simulation_if(M * N * K > 1.2e8)
    g = torch.Generator().manual_seed(M * 7 + N)
    for act, acc, bias, od in ((None, False, True, torch.bfloat16), ("gelu_new", False, True, torch.bfloat16),
                               (None, True, True, torch.float32), (None, False, False, torch.float32),
                               ("gelu", False, True, torch.bfloat16)):
        out, ref = _gemm_case(ops, ops.linear_mfma, M, N, K, torch.bfloat16, act, acc, bias, od, g)
        tol = (1e-2 if od == torch.bfloat16 else 1e-4) * max(1.0, ref.abs().max().item())
        assert (out - ref).abs().max() < tol, (act, acc, bias, od)


@pytest.mark.parametrize("M,N,K", [(1, 4100, 2600), (8, 4800, 1600), helpers.quick(3, 4112, 40), (16, 8192, 72), (17, 6401, 648),
                                   (48, 8190, 1160), (64, 4800, 4616), (9, 5888, 1288), (9, 5889, 1288), (16, 7168, 3080), (16, 7169, 3080),
                                   (4, 5888, 3080), (4, 5889, 3080), (5, 5120, 1288), (5, 5121, 1288), (5, 8192, 4104)])
def test_gemm_one_workgroup_a_compute_unit(ops, M, N, K):
    """Between 4,097 and 8,192 columns: 16 columns a workgroup or up to 32 (17 to 32 here), both sides of the lines between them,
    several rounds of steps in flight, a last step that K cuts; a row has the same bits beside any other rows, so also in either
    kernel; keys and values in the epilogue."""
    g = torch.Generator().manual_seed(M + N)
    for act, acc, bias, od in ((None, False, True, torch.bfloat16), ("gelu_new", False, False, torch.bfloat16), (None, True, True, torch.float32)):
        out, ref = _gemm_case(ops, ops.linear_mfma, M, N, K, torch.bfloat16, act, acc, bias, od, g)
        tol = (1e-2 if od == torch.bfloat16 else 1e-4) * max(1.0, ref.abs().max().item())
        assert (out - ref).abs().max() < tol, (act, acc, bias, od)
    a, w = bf(torch.randn(64, K, generator=g)).to(DEV), bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    rows = lambda lo, hi: ops.linear_mfma(a[lo:hi], w, None, torch.empty(hi - lo, N, device=DEV))
    assert torch.equal(rows(5, 10)[2], rows(0, 64)[7]) and torch.equal(rows(0, 33)[7], rows(4, 20)[3])
    page, D, Hkv = 16, N // 4 // 16 * 4, 2
    if N % 4 == 0 and D % 4 == 0:
        slots = torch.randperm(5 * page, generator=g)[:M].to(torch.int32).to(DEV)
        c1, c2 = (torch.zeros(5, 2, Hkv, page, D, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        ops.linear_mfma(a[:M], w, None, out, kv_cache=c1, slot_map=slots, q_cols=N - 2 * Hkv * D)
        ops.kv_write(out, N - 2 * Hkv * D, N - Hkv * D, c2, slots, Hkv, D)
        assert torch.equal(c1, c2) and bool(c1.any())


@pytest.mark.parametrize("M,N,K", [(1, 1027, 4104), (4, 2048, 8200), helpers.quick(2, 1030, 1032), (3, 50, 1016), (5, 1024, 2048),
                                   helpers.quick(8, 129, 2056), (7, 2048, 6408), (6, 1029, 3080)])
def test_gemm_four_pieces_of_k_side_by_side(ops, M, N, K):
    """Up to 4 rows, or 8 with K from 2,048 on, and up to 2,048 columns: one or two groups of 4 rows and of 4 columns, several rounds of steps,
    a last one that K cuts; a row has the same bits beside any other rows of these kernels, and one that is not finite leaves the others alone."""
    g = torch.Generator().manual_seed(M + N)
    for act, acc, bias, od in ((None, False, True, torch.bfloat16), ("gelu_new", False, False, torch.bfloat16), (None, True, True, torch.float32)):
        out, ref = _gemm_case(ops, ops.linear_mfma, M, N, K, torch.bfloat16, act, acc, bias, od, g)
        tol = (1e-2 if od == torch.bfloat16 else 1e-4) * max(1.0, ref.abs().max().item())
        assert (out - ref).abs().max() < tol, (act, acc, bias, od)
    a, w = bf(torch.randn(8, K, generator=g)).to(DEV), bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    rows = lambda lo, hi: ops.linear_mfma(a[lo:hi], w, None, torch.empty(hi - lo, N, device=DEV))
    most = 8 if K >= 2048 else 4
    whole = rows(0, most)
    assert torch.equal(rows(most - M, most), whole[most - M:]) and torch.equal(rows(1, 2)[0], whole[1])
    a[0, K - 1], a[2, 5] = float("inf"), float("nan")
    assert torch.equal(rows(0, most)[1], whole[1]) and torch.equal(rows(0, most)[3:], whole[3:])


def test_gemm_few_rows_that_lie_far_apart(ops):
    """17 rows of a with 2^27 entries from one to the next (more than 32-bit offsets hold): the same bits as side by side."""
    helpers.skip_in_simulation_if(True, "four gigabytes")
    M, N, K, ld = 17, 4112, 128, (1 << 27) + 64
    far = torch.empty((M - 1) * ld + K, dtype=torch.bfloat16, device=DEV).as_strided((M, K), (ld, 1))
    a, w = (bf(torch.randn(n, K, device=DEV)) for n in (M, N))
    far.copy_(a)
    outs = [ops.linear_mfma(x, w, None, torch.empty(M, N, device=DEV)) for x in (a, far)]
    assert torch.equal(*outs) and bool(outs[0].any())


@pytest.mark.parametrize("M,N,K", [(1, 4800, 1600), (3, 6400, 1600), helpers.quick(2, 4100, 72), (8, 8192, 1304), (16, 4801, 1000), (9, 6000, 768),
                                   helpers.quick(5, 8193, 24), (8, 16384, 1536), (8, 8193, 1544), (1, 8200, 1288), (16, 12800, 1024), (9, 8193, 1032),
                                   (8, 16385, 264), (9, 4801, 1032)])
def test_fused_norm_product_one_workgroup_a_compute_unit(ops, M, N, K):
    """The fused norm and product with up to 32 columns a workgroup, one or two workgroups a compute unit, both sides of the
    lines to 16 columns; parameters in bfloat16 and in 32-bit.  A column has the same bits among fewer columns."""
    g = torch.Generator().manual_seed(M + N)
    x = (torch.randn(M, K, generator=g) * 2 + 1).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    for dt in (torch.bfloat16, torch.float32):
        gw, gb, bias = (torch.randn(n, generator=g).to(dt).to(DEV) for n in (K, K, N))
        out = torch.empty(M, N, device=DEV)
        ops.linear_ln(x, None, M, gw, gb, 1e-5, w, bias, out)
        few = ops.linear_ln(x, None, M, gw, gb, 1e-5, w[:100], bias[:100], torch.empty(M, 100, device=DEV))
        assert torch.equal(out[:, :100], few)
        a = F.layer_norm(x.double(), (K,), gw.double(), gb.double(), 1e-5).to(torch.bfloat16).double()
        ref = a @ w.double().t() + bias.double()
        # (the norm's 32-bit rounding may move an entry of a to the next bfloat16: 2^-8 of one product among K)
        assert (out.double() - ref).abs().max() < 2e-2 * max(1.0, ref.abs().max().item())


@pytest.mark.parametrize("dt", [helpers.quick(torch.bfloat16, mark="simt_a"), torch.float32])
@pytest.mark.parametrize("N,K", [helpers.quick(50, 120, mark="simt_b"), (2304, 512), (1021, 520), (4100, 1024), (4801, 1032), (8190, 1536), (8200, 1544),
                                 helpers.quick(12, 2048, mark="simt_b"), (6401, 1600), (1030, 1792), (2304, 1600), (4801, 1920), (14400, 1536), (16383, 1040),
                                 (2050, 768), (3072, 1024), (3073, 1024), (700, 648), (5121, 896)])
def test_norm_and_product_of_up_to_8_rows(ops, N, K, dt):
    """A wavefront holds one step of 128 k or two, 4 to 8 of them; 4 to 32 columns a workgroup, columns that end inside a group of 4; one group
    of 4 rows or two; a wavefront a row (K up to 256, and most of 5 to 8 rows up to 1,536); rows in any order.  Rows whose mean is a hundred times their spread;
    a row has the same bits beside any others of its kernel, and one that is not finite leaves the others alone."""
    g = torch.Generator().manual_seed(N + K)
    R = 11
    x = (torch.randn(R, K, generator=g) * 3 + torch.arange(R).view(R, 1) * 30.0).to(DEV)
    gw, gb, bias = (torch.randn(n, generator=g).to(dt).to(DEV) for n in (K, K, N))
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    for M in (1, 4, 5, 8):
        rows = torch.randperm(R, generator=g)[:M].to(torch.int32).to(DEV)
        out = ops.linear_ln(x, rows, M, gw, gb, 1e-5, w, bias, torch.empty(M, N, device=DEV))
        a = F.layer_norm(x[rows.long()].double(), (K,), gw.double(), gb.double(), 1e-5).to(torch.bfloat16).double()
        ref = a @ w.double().t() + bias.double()
        # (the norm's 32-bit rounding may move an entry of a to the next bfloat16: 2^-8 of one product among K)
        assert (out.double() - ref).abs().max() < 2e-2 * max(1.0, ref.abs().max().item()), M
        rms = ops.linear_rms(x, rows, M, gw, 1.0, 1e-5, w, bias, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), act="gelu_new")
        xd = x[rows.long()].double()
        a = (xd / (xd.square().mean(1, keepdim=True) + 1e-5).sqrt() * (1.0 + gw.double())).to(torch.bfloat16).double()
        ref = F.gelu(a @ w.double().t() + bias.double(), approximate="tanh")
        assert (rms.double() - ref).abs().max() < 2e-2 * max(1.0, ref.abs().max().item()), M
    whole = ops.linear_ln(x, None, 8, gw, gb, 1e-5, w, bias, torch.empty(8, N, device=DEV))
    few = lambda lo, hi: ops.linear_ln(x[lo:hi].contiguous(), None, hi - lo, gw, gb, 1e-5, w, bias, torch.empty(hi - lo, N, device=DEV))
    four = few(1, 5)
    assert torch.equal(few(2, 3)[0], four[1]) and torch.equal(few(3, 8), whole[3:])
    if K <= 256 or K > 1536 or (640 < K <= 1024 and (N <= 3072 or 4096 < N <= 5120)):      # one kernel
        assert torch.equal(four, whole[1:5])
    x[0, K - 1] = x[1, 3] = float("inf")
    assert torch.equal(few(0, 8)[2:], whole[2:]) and torch.equal(few(1, 5)[1:], four[1:])


@pytest.mark.parametrize("M", [helpers.quick(1), helpers.quick(4, mark="simt_a"), 8])
@pytest.mark.parametrize("K", [helpers.quick(264, mark="simt_b"), 512, 640, 1024, 1160, 1536, 1600, helpers.quick(2048, mark="simt_b")])
def test_norm_statistics_of_rows_that_change_along_k(ops, M, K):
    """Every 128 entries have a mean of their own, far apart beside what they scatter by: the variance is what lies between the parts of a row that the
    wavefronts hold, one or two steps each.  The oracle without that term is 10 tolerances away and more, so a kernel that lost it would be too."""
    g = torch.Generator().manual_seed(M + K)
    part = torch.arange(K) // 128
    x = torch.randn(M, K, generator=g) + 7.0 * ((part * 5 + torch.arange(M).view(M, 1)) % 7)
    gw, gb = torch.randn(K, generator=g) + 2, torch.randn(K, generator=g)
    w = bf(torch.randn(40, K, generator=g) * 0.1)
    out = ops.linear_ln(x.to(DEV), None, M, gw.to(DEV), gb.to(DEV), 1e-5, w.to(DEV), None, torch.empty(M, 40, device=DEV)).double().cpu()
    xd = x.double()
    mean = xd.mean(1, keepdim=True)
    within = sum(((xd[:, part == p] - xd[:, part == p].mean(1, keepdim=True)) ** 2).sum(1, keepdim=True) for p in range(int(part[-1]) + 1)) / K

    def product(variance):
        return ((xd - mean) / torch.sqrt(variance + 1e-5) * gw.double() + gb.double()).to(torch.bfloat16).double() @ w.double().t()

    want = product(((xd - mean) ** 2).mean(1, keepdim=True))
    tol = 2e-3 * max(1.0, want.abs().max().item())
    assert (out - want).abs().max() < tol and (product(within) - want).abs().amax(1).min() > 10 * tol


@pytest.mark.parametrize("M,N,K", [(1600, 2000, 200), (1555, 1999, 320), (2048, 1600, 1600), (1536, 2304, 768), (2048, 2304, 768),
                                   (4096, 768, 3072), (2500, 1600, 2112), (2048, 1600, 6400)])
def test_gemm_tiles_alone_on_their_compute_units(ops, M, N, K):
    """The library's own choice where 128 x 128 tiles would be 140 to 512: a K that a slab cuts and a long K with
    192 to 256 tiles (operands through registers, four slabs in flight: GPT-2 1.5B's proj), whole slabs (operands
    straight into LDS: 128 x 128 tiles for 208 and 216 tiles, GPT-2 1.5B's out-proj among them, and for 260
    tiles with a K above 2,048; 256 x 128 for 288 tiles, GPT-2 124M's q|k|v; 128 x 128 for 192 tiles and a K of 3,072).  What adds into
    the stream goes to the tiles that share k out inside a workgroup instead where K is 3,072 and more and 256 tiles hold it."""
    helpers.skip_in_simulation_if(True)
    g = torch.Generator().manual_seed(M + N + K)
    for act, acc, bias, od in ((None, False, True, torch.bfloat16), ("gelu_new", False, True, torch.bfloat16),
                               (None, True, True, torch.float32), (None, False, False, torch.float32)):
        out, ref = _gemm_case(ops, ops.linear_mfma, M, N, K, torch.bfloat16, act, acc, bias, od, g)
        tol = (1e-2 if od == torch.bfloat16 else 1e-4) * max(1.0, ref.abs().max().item())
        assert (out - ref).abs().max() < tol, (act, acc, bias, od)


@pytest.mark.parametrize("form", ["wide", "wide_256x128", "wide_128x128"])
@pytest.mark.parametrize("M,N,K", [helpers.quick(300, 200, 128), (257, 520, 64), (2048, 1600, 320), (700, 4800, 192)])
def test_gemm_wide_tiles(ops, M, N, K, form):
    """The tiles whose operands go from memory straight into LDS (two stages of a, three of w), in their
    three shapes (256 x 256, 256 x 128, 128 x 128): every epilogue against 64-bit arithmetic, and bit for
    bit what the other tile forms give (all sum over k in ascending steps of 16); edges in M and N, one to
    five slabs."""
    g = torch.Generator().manual_seed(M + N + K)
    wide = lambda *a_, **k_: ops.linear_mfma(*a_, form=form, **k_)
    for act, acc, bias, od in ((None, False, True, torch.bfloat16), ("gelu_new", False, True, torch.bfloat16),
                               ("gelu", False, False, torch.bfloat16), (None, True, True, torch.float32),
                               (None, False, False, torch.float32), ("silu", False, True, torch.bfloat16)):
        out, ref = _gemm_case(ops, wide, M, N, K, torch.bfloat16, act, acc, bias, od, g)
        tol = (1e-2 if od == torch.bfloat16 else 1e-4) * max(1.0, ref.abs().max().item())
        assert (out - ref).abs().max() < tol, (act, acc, bias, od)
    a = bf(torch.randn(M, K, generator=g) * 0.5).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.2).to(DEV)
    b = bf(torch.randn(N, generator=g)).to(DEV)
    for od, acc in ((torch.bfloat16, False), (torch.float32, True)):
        o1 = torch.full((M, N), 0.25, device=DEV, dtype=od)
        o2 = o1.clone()
        ops.linear_mfma(a, w, b, o1, None, acc, form=form)
        ops.linear_mfma(a, w, b, o2, None, acc)
        assert torch.equal(o1, o2), (od, acc)
    with pytest.raises(ops.KernelError, match="multiple of 64"):
        ops.linear_mfma(a[:, :K - 8].contiguous(), w[:, :K - 8].contiguous(), b, o1, form=form)


@pytest.mark.parametrize("M", [1, 5, helpers.quick(9), 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("inner,K", [helpers.quick(1030, 72), (2048, 768), (2752, 1024), (1100, 2056), (5000, 2048)])
def test_gated_products_of_few_rows(ops, M, inner, K):
    """The gate and up products with their activation in one kernel, against 64 bits: a rounding to bfloat16 of the result and the
    hardware's exp2 and reciprocal in between; the last workgroup's columns cut, rows that are not whole tiles, both numbers of
    wavefronts.  What it does not take goes to the two kernels."""
    g = torch.Generator().manual_seed(M + inner + K)
    a = bf(torch.randn(M, K, generator=g) * 0.5).to(DEV)
    w = bf(torch.randn(2 * inner, K, generator=g) * (1.0 / K ** 0.5)).to(DEV)
    takes = bool(ops._lib().da_gemm_gated_takes(M, inner, K))
    # (above 16 rows: with a workgroup for every compute unit, and no more columns than few rows may have)
    assert takes == (M <= 16 or inner == 2048 or (inner == 5000 and M <= 32))
    wide = torch.zeros(M, inner + 8, dtype=torch.bfloat16, device=DEV)
    for act, limit in (("silu", 0.0), ("gelu_new", 0.0), ("glu_capped", 1.5)):
        mid = wide[:, :inner]
        if not takes:
            with pytest.raises(ops.KernelError, match="not taken"):
                ops.linear_gated(a, w, mid, act, limit)
            return
        ops.linear_gated(a, w, mid, act, limit)
        z = a.double().cpu() @ w.double().cpu().t()
        gate, up = z[:, :inner], z[:, inner:]
        if act == "glu_capped":
            gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
            ref = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
        else:
            ref = (F.silu(gate) if act == "silu" else F.gelu(gate, approximate="tanh")) * up
        assert ((mid.double().cpu() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all(), act
        assert not wide[:, inner:].any()


@pytest.mark.simt_quick
def test_which_products_into_the_stream_share_k_out_inside_a_workgroup(ops):
    """The tiles of 128 x 64 (4) and 128 x 128 (3) where they were measured ahead, and not (-1) where others are level or ahead."""
    choice = ops._lib().da_gemm_deep_choice
    for M, N, K, want in ((1624, 1024, 1024, 4), (1624, 1024, 4096, 4), (2048, 768, 3072, 4), (593, 2560, 1152, 4), (1549, 1152, 2048, 4), (1535, 1216, 1024, 4),
                          (2048, 1600, 6400, 3), (4096, 1024, 4096, 3), (1300, 1536, 3072, 3), (354, 5120, 1024, -1), (700, 2048, 1024, -1), (2600, 768, 1024, -1),
                          (2600, 768, 3072, -1), (3104, 640, 1280, -1), (1024, 1024, 4096, -1), (4096, 1024, 2048, -1), (4096, 2048, 4096, -1), (1624, 1024, 4104, -1)):
        assert choice(M, N, K) == want, (M, N, K)


@pytest.mark.simt_quick
def test_profiler_names_the_tiles_of_a_product(ops):
    """One name each for the products into the stream that share k out inside a workgroup, the other tiles with operands straight into LDS and
    the rest; an activation keeps a product out of the first."""
    f32, bf16 = torch.empty(0), torch.empty(0, dtype=torch.bfloat16)
    for M, N, K, act, acc, out, want in ((1624, 1024, 4096, None, True, f32, "deep"), (2048, 1600, 6400, None, True, f32, "deep"),
                                         (1300, 1536, 3072, "gelu_new", True, f32, "tile"), (2048, 4800, 1600, None, False, bf16, "wide"),
                                         (4096, 1024, 4096, None, False, f32, "wide"), (2048, 6400, 1600, "gelu_new", False, bf16, "wide"),
                                         (2048, 6400, 1600, "gelu_new", False, f32, "tile"), (2048, 4800, 1608, None, False, bf16, "tile"), (300, 96, 200, None, True, f32, "tile")):
        assert ops._tile_name(M, N, K, act, acc, out) == "product_" + want, (M, N, K, act, acc)


@pytest.mark.parametrize("M,N,K", [helpers.quick(65, 8256, 1024), (1300, 1536, 3072)])
def test_products_into_the_stream_keep_their_activation(ops, M, N, K):
    """Sizes that go to each of the two tiles that share k out inside a workgroup, which have no activation: with one the product is
    another kernel's, without one theirs."""
    helpers.skip_in_simulation_if(M * N * K > 1e9)
    g = torch.Generator().manual_seed(M + N)
    for act in ("gelu_new", None):
        out, ref = _gemm_case(ops, ops.linear, M, N, K, torch.bfloat16, act, True, True, torch.float32, g)
        assert (out - ref).abs().max() < 1e-4 * max(1.0, ref.abs().max().item()), act


@pytest.mark.parametrize("form", ["deep_128x128", "deep_128x64"])
@pytest.mark.parametrize("M,N,K", [helpers.quick(130, 70, 1024), (128, 128, 1088), (257, 200, 1152), (640, 1600, 6400), (1624, 1024, 4096)])
def test_gemm_deep_tiles(ops, M, N, K, form):
    """The tiles that add into the stream with k shared out over the wavefronts of a workgroup (two and four a position), five and six
    slabs ahead: an odd and an even number of slabs, edges in M and N.  A sum of K products of bfloat16 in 32-bit, in 16 or more
    partial sums of a product's own k, is off by less than K / 16 roundings of 2^-24 of the sum of absolute values."""
    g = torch.Generator().manual_seed(M + N + K)
    a = bf(torch.randn(M, K, generator=g) * 0.5).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.2).to(DEV)
    x = torch.randn(M, N, generator=g).to(DEV)
    bound = (a.abs().float() @ w.abs().float().t()) * (K / 16 * 2.0 ** -24) + 1e-5
    ref = x.double().cpu() + a.double().cpu() @ w.double().cpu().t()
    for bias in (None, bf(torch.randn(N, generator=g)).to(DEV), torch.randn(N, generator=g).to(DEV)):
        wide = torch.zeros(M, N + 12, device=DEV)
        out = wide[:, 4:N + 4] if N % 4 == 0 else wide[:, 3:N + 3]
        out.copy_(x)
        ops.linear_mfma(a, w, bias, out, None, True, form=form)
        want = ref if bias is None else ref + bias.double().cpu()
        assert ((out.double().cpu() - want).abs() <= bound.double().cpu()).all()
        assert not wide[:, N + 4:].any() and not wide[:, :3].any()
        if (M, form) == (1624, "deep_128x64"):       # the library's own choice there
            auto = x.clone()
            ops.linear_mfma(a, w, bias, auto, None, True)
            assert torch.equal(auto, out)
    with pytest.raises(ops.KernelError, match="adds into the stream"):
        ops.linear_mfma(a, w, None, torch.empty(M, N, device=DEV), form=form)


@pytest.mark.parametrize("form", ["wide", "wide_256x128", "wide_128x128"])
@pytest.mark.parametrize("M", [helpers.quick(300), 1000])
def test_gemm_wide_tiles_write_keys_and_values(ops, M, form):
    g = torch.Generator().manual_seed(M)
    Hq, Hkv, D, page, K = 5, 3, 48, 16, 128
    N = (Hq + 2 * Hkv) * D
    n_pages = (M + page - 1) // page + 2
    a = bf(torch.randn(M, K, generator=g)).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    bias = bf(torch.randn(N, generator=g)).to(DEV)
    perm = torch.randperm(n_pages * page, generator=g)[:M].to(torch.int32)
    perm[M // 2] = -1
    runs = torch.cat([torch.arange(16, 16 + M // 2), torch.arange(16 + M // 2 + 19, 16 + M // 2 + 19 + M - M // 2)]).to(torch.int32)
    runs[M // 4] = -1
    for order in (perm, runs):
        slots = order.to(DEV)
        c1 = torch.zeros(n_pages + 2, 2, Hkv, page, D, dtype=torch.bfloat16, device=DEV)
        c2 = torch.zeros_like(c1)
        out1 = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        out2 = torch.empty_like(out1)
        ops.linear_mfma(a, w, bias, out1, kv_cache=c1, slot_map=slots, q_cols=Hq * D, form=form)
        ops.linear_mfma(a, w, bias, out2)
        ops.kv_write(out2, Hq * D, (Hq + Hkv) * D, c2, slots, Hkv, D)
        assert torch.equal(out1, out2)
        assert torch.equal(c1, c2) and c1.abs().sum() > 0


@pytest.mark.simt_quick
@pytest.mark.parametrize("form", ["auto", "wide", "wide_256x128", "wide_128x128"])
@pytest.mark.parametrize("M", [512, 517])
def test_product_writes_values_of_prompts_of_odd_lengths(ops, M, form):
    """More than 512 rows of several sequences, each from any place of a page on: groups of 4 places that begin with
    each row of a piece of 32, pieces with rows of two sequences, and rows without a place at the start, in the middle
    and at the end of a group.  512 rows take the way of few rows."""
    g = torch.Generator().manual_seed(M)
    Hq, Hkv, D, page, K = 1, 2, 24, 16, 64
    N = (Hq + 2 * Hkv) * D
    a, w, bias = (bf(torch.randn(*s, generator=g)).to(DEV) for s in ((M, K), (N, K), (N,)))
    places, page0 = [], 1
    for first, n in ((0, 64), (1, 95), (2, 97), (3, 94), (5, 33), (0, 2), (6, 70), (0, M - 455)):
        places += range(page0 * page + first, page0 * page + first + n)
        page0 += (first + n) // page + 2
    slots = torch.tensor(places, dtype=torch.int32)
    assert slots.numel() == M
    for r in (96, 130, 195, 260, 393, M - 1):
        slots[r] = -1
    slots = slots.to(DEV)
    c1 = torch.zeros(page0 + 1, 2, Hkv, page, D, dtype=torch.bfloat16, device=DEV)
    c2 = torch.zeros_like(c1)
    out1, out2 = (torch.empty(M, N, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.linear_mfma(a, w, bias, out1, kv_cache=c1, slot_map=slots, q_cols=Hq * D, form=form)
    ops.linear_mfma(a, w, bias, out2)
    ops.kv_write(out2, Hq * D, (Hq + Hkv) * D, c2, slots, Hkv, D)
    assert torch.equal(out1, out2)
    assert torch.equal(c1, c2) and c1.abs().sum() > 0


@pytest.mark.simt_quick
@pytest.mark.parametrize("M", [20, 200])
def test_gemm_into_rows_longer_than_the_result(ops, M):
    """The output's rows are longer than N (a view of a wider matrix): the tile kernel stores whole
    16-byte pieces up to the last one that N cuts, which goes out entry by entry; what lies behind
    column N is not touched, with a store, a 32-bit store and +=."""
    g = torch.Generator().manual_seed(M)
    N, K, LD = 1030, 96, 1040
    a = bf(torch.randn(M, K, generator=g) * 0.5).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.2).to(DEV)
    b = bf(torch.randn(N, generator=g)).to(DEV)
    ref = a.double() @ w.double().t() + b.double()
    for od, acc in ((torch.bfloat16, False), (torch.float32, False), (torch.float32, True)):
        big = torch.full((M, LD), 7.0, device=DEV, dtype=od)
        out = big[:, :N]
        ops.linear_mfma(a, w, b, out, None, acc)
        want = ref + (7.0 if acc else 0.0)
        tol = (1e-2 if od == torch.bfloat16 else 1e-4) * max(1.0, want.abs().max().item())
        assert (out.double() - want).abs().max() < tol, (od, acc)
        assert torch.equal(big[:, N:], torch.full((M, LD - N), 7.0, device=DEV, dtype=od)), (od, acc)


@pytest.mark.simt_quick
def test_gemm_rows_do_not_depend_on_the_batch(ops):
    """A row's result is the same, bit for bit, whatever other rows share the call, as long as the call
    takes the same kernel form (block tiles; 16x16x32 products up to 64 rows; of four pieces of k up to 4
    rows and 2,048 columns); between forms it differs by the rounding of 32-bit sums at most."""
    g = torch.Generator().manual_seed(3)
    K, N = 768, 300
    a = bf(torch.randn(200, K, generator=g)).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)

    def rows(lo, hi, dtype=torch.bfloat16):
        out = torch.empty(hi - lo, N, device=DEV, dtype=dtype)
        ops.linear_mfma(a[lo:hi].contiguous(), w, None, out)
        return out

    full = rows(0, 200)
    assert torch.equal(rows(60, 150), full[60:150])                 # block tiles
    small = rows(0, 64)
    assert torch.equal(rows(3, 23)[7], small[10])                   # 16x16x32: 20 rows, 64 rows
    assert torch.equal(rows(4, 12)[6], small[10])                   # ... 8 rows
    assert torch.equal(rows(10, 11)[0], rows(8, 12)[2])             # four pieces of k: 1 row, 4 rows
    assert torch.equal(rows(10, 13)[0], rows(10, 11)[0])            # ... 3 rows
    exact = a[10].double() @ w.double().t()
    scale = exact.abs().max().item()
    forms = [rows(10, 11, torch.float32)[0], rows(0, 64, torch.float32)[10], rows(0, 200, torch.float32)[10]]
    for f in forms:
        assert (f.double() - exact).abs().max() < 2e-6 * scale


@pytest.mark.simt_quick
def test_gemm_refuses_what_it_cannot_take(ops):
    a = torch.zeros(4, 12, device=DEV, dtype=torch.bfloat16)
    w = torch.zeros(8, 12, device=DEV, dtype=torch.bfloat16)
    out = torch.zeros(4, 8, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ops.KernelError, match="multiples of 8"):
        ops.linear_mfma(a, w, None, out)
    ops.linear(a, w, None, out)                     # the dispatcher sends it to the plain kernel
    with pytest.raises(ops.KernelError):
        ops.linear_ref(a, w, None, torch.zeros(4, 9, device=DEV, dtype=torch.bfloat16))
    with pytest.raises(ops.KernelError, match="float32 output"):
        ops.linear_ref(a, w, None, out, None, True)


# ----------------------------------------------------------------------------- paged attention
class PagedCase:
    """Sequences with their keys and values scattered over a NaN-filled pool."""

    def __init__(self, lens, new, Hq, Hkv, D, page, dtype, seed, scale_boost=None):
        g = torch.Generator().manual_seed(seed)
        self.lens, self.new, self.Hq, self.Hkv, self.D, self.page = lens, new, Hq, Hkv, D, page
        S = len(lens)
        n_pages = sum(-(-n // page) for n in lens) + 5
        perm = torch.randperm(n_pages, generator=g).tolist()
        self.cache = torch.full((n_pages, 2, Hkv, page, D), float("nan"), dtype=dtype, device=DEV)
        max_blocks = max(-(-n // page) for n in lens)
        bt = torch.full((S, max_blocks), -1, dtype=torch.int32)
        self.k, self.v, self.q = [], [], []
        for s, n in enumerate(lens):
            k = torch.randn(n, Hkv * D, generator=g).to(dtype)
            v = torch.randn(n, Hkv * D, generator=g).to(dtype)
            q = torch.randn(new[s], Hq * D, generator=g).to(dtype)
            if scale_boost is not None:      # one far key stands out for the last query
                far, boost = scale_boost
                q[-1] *= boost
                qv = q[-1].float().view(Hq, D)[:: Hq // Hkv]
                k[far] = (qv / qv.norm(dim=1, keepdim=True) * 8.0).reshape(-1).to(dtype)
            self.k.append(k); self.v.append(v); self.q.append(q)
            for j in range(-(-n // page)):
                bt[s, j] = perm.pop()
        self.bt = bt.to(DEV)
        # fill through the engine's own write kernel
        from deliverance_amd.kernels import ops as o
        for s, n in enumerate(lens):
            qkv = torch.cat([torch.zeros(n, Hq * D, dtype=dtype), self.k[s], self.v[s]], dim=1).to(DEV)
            slots = torch.tensor([int(bt[s, pos // page]) * page + pos % page for pos in range(n)], dtype=torch.int32, device=DEV)
            o.kv_write(qkv, Hq * D, Hq * D + Hkv * D, self.cache, slots, Hkv, D)
        self.qcat = torch.cat(self.q).to(DEV)
        starts = np.cumsum([0] + list(new))
        self.q_start = torch.tensor(starts, dtype=torch.int32, device=DEV)
        self.seq_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
        self.seq_of = torch.tensor([s for s, n in enumerate(new) for _ in range(n)], dtype=torch.int32, device=DEV)
        self.pos = torch.tensor([lens[s] - new[s] + i for s in range(S) for i in range(new[s])], dtype=torch.int32, device=DEV)

    def plain(self, scale, window):
        outs = []
        for s in range(len(self.lens)):
            o = P.causal_attention(self.q[s].double().numpy(), self.k[s].double().numpy(), self.v[s].double().numpy(),
                                   self.Hq, scale, window=window, n_kv_head=self.Hkv, past=self.lens[s] - self.new[s])
            outs.append(o)
        return np.concatenate(outs)


ATT_TOL = {torch.float32: 2e-5, torch.bfloat16: 2e-2}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,D,page,window", [helpers.quick(4, 4, 16, 16, None), (6, 2, 48, 16, None), helpers.quick(2, 1, 80, 32, 37),
                                                  (3, 3, 128, 64, None), (5, 5, 64, 16, 100)])
def test_attention_plain_kernel(ops, dtype, Hq, Hkv, D, page, window):
    case = PagedCase(lens=[70, 5, 131, 64], new=[70, 1, 9, 2], Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=dtype, seed=D)
    out = torch.empty_like(case.qcat)
    scale = 0.7 / math.sqrt(D)
    ops.attention_ref(case.qcat, case.cache, case.bt, case.seq_of, case.pos, Hq, scale, window, out)
    assert np.abs(out.double().cpu().numpy() - case.plain(scale, window)).max() < ATT_TOL[dtype]


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [helpers.quick(4, 4, 16, 16, None), (6, 2, 48, 16, None), helpers.quick(2, 1, 80, 32, 37),
                                                  (3, 3, 128, 64, None), (12, 12, 64, 16, None), (5, 5, 64, 16, 100), (2, 1, 96, 16, 70),
                                                  (2, 2, 112, 16, None)])
def test_attention_32bit_on_the_matrix_cores(ops, Hq, Hkv, D, page, window):
    """Portions and one-token sequences in one launch, chunk edges, a padding sequence; a row has the same bits however its
    portion is cut."""
    lens, new = [70, 5, 131, 64, 1, 65, 600, 129], [70, 1, 9, 17, 1, 1, 33, 129]
    case = PagedCase(lens=lens, new=new, Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=torch.float32, seed=D)
    scale = 0.7 / math.sqrt(D)
    out = torch.full_like(case.qcat, 7.0)
    ops.attention_f32(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, len(lens), max(new), Hq, scale, window, out)
    assert np.abs(out.double().cpu().numpy() - case.plain(scale, window)).max() < ATT_TOL[torch.float32]
    # the last 5 rows of the last sequence alone, then a sequence of length 0
    one = torch.full((6, Hq * D), 7.0, device=DEV)
    q = torch.cat([case.qcat[-5:], case.qcat[:1]])
    bt = torch.cat([case.bt[-1:], torch.full_like(case.bt[:1], -1)])
    ops.attention_f32(q, case.cache, bt, torch.tensor([0, 5, 6], dtype=torch.int32, device=DEV),
                      torch.tensor([129, 0], dtype=torch.int32, device=DEV), 2, 5, Hq, scale, window, one)
    assert torch.equal(one[:5], out[-5:]) and not bool(one[5].any())


@pytest.mark.simt_quick
def test_attention_32bit_of_a_cache_that_is_not_aligned(ops):
    """Rows of q or a cache whose first byte is no multiple of 16: the plain kernel's; fewer rows in out than in q: refused."""
    from types import SimpleNamespace
    D, page, Hq = 16, 16, 2
    case = PagedCase(lens=[33, 5], new=[20, 1], Hq=Hq, Hkv=1, D=D, page=page, dtype=torch.float32, seed=3)
    ctx = SimpleNamespace(block_tables=[case.bt], n_decode=0, n_seqs=2, max_query_len=20, q_start=case.q_start, seq_lens=case.seq_lens,
                          seq_of_token=case.seq_of, positions=case.pos, seq_lens_host=[33, 5], q_start_host=[0, 20, 21])
    cache = torch.empty(case.cache.numel() + 1, device=DEV)[1:].view(case.cache.shape)
    cache.copy_(case.cache)
    qs = torch.empty(21, Hq * D + 1, device=DEV)[:, 1:]
    qs.copy_(case.qcat)
    want = case.plain(0.3, None)
    for q, c in ((case.qcat, case.cache), (case.qcat, cache), (qs, case.cache)):
        out = torch.full_like(case.qcat, 7.0)
        ops.paged_attention(ctx, q, c, 0, Hq, 0.3, None, out)
        assert np.abs(out.double().cpu().numpy() - want).max() < ATT_TOL[torch.float32]
    with pytest.raises(ops.KernelError, match="row|q/out"):
        ops.paged_attention(ctx, case.qcat, case.cache, 0, Hq, 0.3, None, out[:20])


def _attention_64(q, k, v, past, scale, window):
    """One head in 64 bits, row by row: a value whose weight is zero is not looked at, scores without a number or of plus
    infinity (or of minus infinity alone) leave no number."""
    out = np.zeros((q.shape[0], v.shape[1]))
    with np.errstate(all="ignore"):
        for i in range(q.shape[0]):
            lo = max(0, past + i - window + 1) if window else 0
            s = (k[lo:past + i + 1] @ q[i]) * scale
            e = np.exp(s - s.max())
            seen = e != 0.0
            out[i] = (e[seen, None] * v[lo:past + i + 1][seen]).sum(0) / e.sum()
    return out


@pytest.mark.simt_quick
@pytest.mark.parametrize("window", [None, 20])
def test_attention_32bit_with_numbers_that_are_not_finite(ops, window):
    """Infinite and missing numbers in queries, keys and values: they reach the rows that see them with a weight and no
    other row, though 16 rows and 64 keys share a tile.  (Every row is compared, bound as for finite numbers.)"""
    inf, nan = float("inf"), float("nan")
    D, page, T, past = 16, 16, 40, 90
    n = past + T
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(n, D, generator=g) for _ in range(3))
    q = q[:T].abs() + 0.1
    v[past + 9, 3], v[past + 21, 4], v[past + 30, 5] = inf, nan, -inf     # seen by the rows behind them only
    k[past + 12] = -inf                                                  # a score of minus infinity: no weight
    v[past + 12] = nan
    k[past + 35, 2] = nan                                                # rows from 35 on: no number
    k[64:64 + 20] = -inf                                                 # with the window some rows' first chunk is this alone
    q[2, 7] = nan
    cache = torch.full((12, 2, 1, page, D), nan)
    bt = torch.tensor([[3, 7, 1, 9, 0, 4, 8, 2, 5]], dtype=torch.int32)
    for j in range(n):
        cache[bt[0, j // page], 0, 0, j % page] = k[j]
        cache[bt[0, j // page], 1].view(D, page)[:, j % page] = v[j]
    out = torch.full((T, D), 7.0, device=DEV)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ops.attention_f32(q.to(DEV), cache.to(DEV), bt.to(DEV), i32(0, T), i32(n), 1, T, 1, 0.2, window, out)
    want = _attention_64(q.double().numpy(), k.double().numpy(), v.double().numpy(), past, 0.2, window)
    got = out.double().cpu().numpy()
    assert np.isnan(want).any() and np.isposinf(want).any() and np.isfinite(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fin = np.isfinite(want)
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]) and np.abs(got[fin] - want[fin]).max() < ATT_TOL[torch.float32]


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [helpers.quick(4, 4, 16, 16, None), (6, 2, 48, 16, None), helpers.quick(2, 1, 80, 32, 37),
                                                  (3, 3, 128, 64, None), (12, 12, 64, 16, None), (5, 5, 64, 16, 100),
                                                  helpers.quick(2, 2, 256, 16, None), (25, 25, 64, 32, 70)])
def test_attention_decode_kernel(ops, Hq, Hkv, D, page, window):
    lens = [1, 2, 63, 64, 65, 300, 129, 17, 1000]
    case = PagedCase(lens=lens, new=[1] * len(lens), Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=torch.bfloat16, seed=D + 1)
    out = torch.empty_like(case.qcat)
    scale = 0.7 / math.sqrt(D)
    ops.attention_decode(case.qcat, case.cache, case.bt, case.seq_lens, len(lens), Hq, scale, window, out)
    got = out.double().cpu().numpy()
    assert np.isfinite(got).all()
    assert np.abs(got - case.plain(scale, window)).max() < ATT_TOL[torch.bfloat16]


@pytest.mark.simt_quick
@pytest.mark.parametrize("D", [16, 48, 80, 144])
def test_attention_decode_with_infinite_keys_and_values(ops, D):
    """A key of minus infinity in some dimension has no weight (head sizes that are no multiple of 32 fill the matrix
    instruction's depth with zeros, which may not meet it), an infinite value stands in the result."""
    inf, page, n = float("inf"), 16, 100
    g = torch.Generator().manual_seed(D)
    q, k, v = (bf(torch.randn(m, D, generator=g)) for m in (1, n, n))
    q = q.abs() + 0.25
    k[70, 1] = k[71, 7] = k[3, 0] = k[60, 20 % D] = k[99, D - 1] = k[40, D - 9] = -inf
    v[50, 2], v[20, D - 1] = -inf, inf
    cache = torch.full((7, 2, 1, page, D), float("nan"), dtype=torch.bfloat16)
    for j in range(n):
        cache[j // page, 0, 0, j % page] = k[j]
        cache[j // page, 1].view(D, page)[:, j % page] = v[j]
    out = torch.empty(1, D, dtype=torch.bfloat16, device=DEV)
    ops.attention_decode(q.to(DEV), cache.to(DEV), torch.arange(7, dtype=torch.int32, device=DEV).view(1, 7),
                         torch.tensor([n], dtype=torch.int32, device=DEV), 1, 1, 0.2, None, out)
    want = _attention_64(q.double().numpy(), k.double().numpy(), v.double().numpy(), n - 1, 0.2, None)
    got = out.double().cpu().numpy()
    fin = np.isfinite(want)
    assert fin.sum() == D - 2 and np.array_equal(got[~fin], want[~fin])
    assert np.abs(got[fin] - want[fin]).max() < ATT_TOL[torch.bfloat16]


@pytest.mark.simt_quick
@pytest.mark.parametrize("rel", [False, True])
@pytest.mark.parametrize("D,page,window", [(64, 16, None), (64, 8, 75), (128, 64, 75), (32, 32, None), (48, 16, 75), (80, 8, None), (16, 16, None)])
def test_attention_decode_scores_of_an_infinite_keys_neighbours(ops, D, page, window, rel):
    """The scores of four keys that follow each other by fours are sums over all of their dimensions with zeros in the place of the
    others' (attn_decode.hip): a key of minus infinity takes its own weight and nobody else's, in each of the four places, in whole
    chunks and in the one that a window or the length cuts; also with a bias by distance."""
    inf, n = float("inf"), 150
    g = torch.Generator().manual_seed(D + page)
    q, k, v = (bf(torch.randn(m, D, generator=g)) for m in (1, n, n))
    q = q.abs() + 0.25
    hit = torch.tensor([0, 5, 10, 15, 64 + 3, 64 + 17, 64 + 42, 128 + 20, n - 1])
    k[hit, (hit * 7) % D] = -inf
    pages = -(-n // page)
    cache = torch.full((pages, 2, 1, page, D), float("nan"), dtype=torch.bfloat16)
    for j in range(n):
        cache[j // page, 0, 0, j % page] = k[j]
        cache[j // page, 1].view(D, page)[:, j % page] = v[j]
    out = torch.empty(1, D, dtype=torch.bfloat16, device=DEV)
    args = (q.to(DEV), cache.to(DEV), torch.arange(pages, dtype=torch.int32, device=DEV).view(1, pages),
            torch.tensor([n], dtype=torch.int32, device=DEV), 1, 1, 0.2, window)
    lo = n - window if window else 0
    s = (k[lo:].double() @ q[0].double()) * 0.2
    if rel:
        bias = torch.randn(1, 40, generator=g)
        s = s + bias[0, torch.arange(n - 1 - lo, -1, -1).clamp(max=39)].double()
        ops.attention_decode_rel(*args, bias.to(DEV), 0.0, 0, out)
    else:
        ops.attention_decode(*args, out)
    want = torch.softmax(s, 0) @ v[lo:].double()
    assert bool(torch.isfinite(want).all()) and (out[0].double().cpu() - want).abs().max() < ATT_TOL[torch.bfloat16]


@pytest.mark.simt_quick
@pytest.mark.parametrize("D", [16, 64, 80, 144])
def test_attention_decode_keeps_the_weights_32_bits(ops, D):
    """Pairs of keys whose weights differ by 2^-12 and whose values, 65,536 and its negative, nearly cancel: the result is what
    the weights' low bits say.  Root mean square of the error: the result's rounding to bfloat16 (at most 2^-9 of it) and 2e-3,
    about six times what the same sums in 32 bits lose; weights of 16 bits lose more than twice the bound, of 8 a
    thousand times."""
    A, n, page, scale = 65536.0, 200, 16, 0.125
    g = torch.Generator().manual_seed(D)
    q, k = bf(torch.randn(1, D, generator=g)), bf(torch.randn(n, D, generator=g) * 0.5)
    q[0, 0] = 2.0 ** -6
    k[1::2] = k[0::2]
    k[0::2, 0] = 0.0
    k[1::2, 0] = bf(torch.randn(n // 2, generator=g).sign() * 0.125)
    v = torch.randn(n // 2, D, generator=g).sign() * A
    v = bf(torch.stack([v, -v], 1).reshape(n, D))
    s = (k.double() @ q[0].double()) * scale
    e = torch.exp(s - s.max())
    result = lambda weights: (weights @ v.double()) / e.sum()
    want = result(e)
    rms = lambda x: x.square().mean().sqrt().item()
    bound = 2.0 ** -9 * rms(want) + 2e-3
    high = bf(e).double()
    assert rms(result(high) - want) > 100 * bound and rms(result(high + bf(e - high).double()) - want) > 2 * bound
    cache = torch.full((13, 2, 1, page, D), float("nan"), dtype=torch.bfloat16)
    for j in range(n):
        cache[j // page, 0, 0, j % page] = k[j]
        cache[j // page, 1].view(D, page)[:, j % page] = v[j]
    out = torch.empty(1, D, dtype=torch.bfloat16, device=DEV)
    ops.attention_decode(q.to(DEV), cache.to(DEV), torch.arange(13, dtype=torch.int32, device=DEV).view(1, 13),
                         torch.tensor([n], dtype=torch.int32, device=DEV), 1, 1, scale, None, out)
    assert rms(out[0].double().cpu() - want) < bound


@pytest.mark.parametrize("n_splits", [2, helpers.quick(3, mark="simt_a"), 7, 16])
@pytest.mark.parametrize("Hq,Hkv,D,page,window", [helpers.quick(2, 2, 64, 16, None, mark="simt_b"), (4, 2, 48, 32, None),
                                                  helpers.quick(1, 1, 128, 64, 700, mark="simt_b"), (3, 3, 16, 16, 90)])
def test_attention_decode_with_keys_split_over_workgroups(ops, Hq, Hkv, D, page, window, n_splits):
    """Every (sequence, head) pair's keys in ``n_splits`` shares with a merge in a fixed order: shares
    that hold nothing (short sequences, a window that has passed them), one key, a share's first and
    last key, sequences that end at a share's edge."""
    width = 2100                                                   # keys the block table spans
    span = -(-(-(-width // page) * page) // n_splits // 64) * 64    # what the kernel gives a share
    lens = [1, 2, 63, span, span + 1, 2 * span - 1 if 2 * span - 1 <= width else width, 1030, width, 700]
    case = PagedCase(lens=lens, new=[1] * len(lens), Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=torch.bfloat16, seed=D + n_splits)
    assert case.bt.shape[1] == -(-width // page)
    scale = 0.7 / math.sqrt(D)
    out = torch.full_like(case.qcat, float("nan"))
    ws = torch.full((ops.decode_workspace_floats(len(lens), Hq, D, n_splits),), float("nan"), device=DEV)
    ops.attention_decode(case.qcat, case.cache, case.bt, case.seq_lens, len(lens), Hq, scale, window, out, n_splits, ws)
    got = out.double().cpu().numpy()
    assert np.isfinite(got).all()
    assert np.abs(got - case.plain(scale, window)).max() < ATT_TOL[torch.bfloat16]
    one = torch.empty_like(case.qcat)
    ops.attention_decode(case.qcat, case.cache, case.bt, case.seq_lens, len(lens), Hq, scale, window, one)
    assert (out.float() - one.float()).abs().max() < 2e-2          # the two kernels differ by rounding only
    with pytest.raises(ops.KernelError, match="workspace"):
        ops.attention_decode(case.qcat, case.cache, case.bt, case.seq_lens, len(lens), Hq, scale, window, out, n_splits, ws[:10])


@pytest.mark.parametrize("where", ["first", "share_end", helpers.quick("share_start"), "second_share_end", "last", "window_edge"])
@pytest.mark.parametrize("D,page,window,n_splits", [helpers.quick(64, 16, None, 3), (144, 32, None, 2), (64, 16, 700, 4), (32, 64, 1500, 16)])
def test_attention_decode_split_sees_one_far_key(ops, D, page, window, n_splits, where):
    """One key among 2,100 carries nearly all the weight of the last query: a share's first or last key,
    the sequence's first or last, or the oldest key that the window still holds.  Random keys alone give
    near-uniform weights, under which a lost key moves the result by a thousandth."""
    n = 2100
    span = -(-(-(-n // page) * page) // n_splits // 64) * 64
    far = {"first": 0, "share_end": span - 1, "share_start": span, "second_share_end": min(2 * span, n) - 1, "last": n - 1,
           "window_edge": n - (window or n)}[where]
    Hq, Hkv = 2, 1
    case = PagedCase(lens=[n], new=[1], Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=torch.bfloat16, seed=D + far, scale_boost=(far, 3.0))
    scale = 0.7 / math.sqrt(D)
    want = case.plain(scale, window)
    seen = window is None or far >= n - window
    if seen:      # the far key's value is the answer, nearly
        assert np.abs(want[0, :D] - case.v[0][far].double().numpy()[:D]).max() < 0.1
    out = torch.full_like(case.qcat, float("nan"))
    ws = torch.full((ops.decode_workspace_floats(1, Hq, D, n_splits),), float("nan"), device=DEV)
    ops.attention_decode(case.qcat, case.cache, case.bt, case.seq_lens, 1, Hq, scale, window, out, n_splits, ws)
    assert np.abs(out.double().cpu().numpy() - want).max() < ATT_TOL[torch.bfloat16], (where, far)


@pytest.mark.simt_quick
def test_when_decode_attention_splits_its_keys(ops):
    assert ops.decode_splits(1, 12, 64, 16) == 1                   # 1,024 keys: one share
    assert ops.decode_splits(1, 12, 256, 16) == 4                  # 4,096 keys, 12 pairs: shares of 1,024
    assert ops.decode_splits(8, 25, 256, 16) == 2                  # 200 pairs: two shares fill the chip
    assert ops.decode_splits(64, 12, 256, 16) == 1                 # 768 pairs fill it alone
    assert ops.decode_splits(1, 1, 4096, 16) == 32                 # never more than 32


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [(4, 4, 16, 16, None), helpers.quick(6, 2, 48, 16, None), helpers.quick(2, 1, 80, 32, 37),
                                                  (3, 3, 128, 64, None), (12, 12, 64, 16, None), (5, 5, 64, 16, 100),
                                                  (2, 2, 256, 16, None), (2, 2, 240, 16, None), helpers.quick(3, 1, 64, 32, 200)])
def test_attention_prefill_kernel(ops, Hq, Hkv, D, page, window):
    lens = [70, 200, 131, 64, 2, 300, 513]
    new = [70, 9, 131, 2, 2, 129, 260]            # whole prompts, short portions after a long past, tiles' edges
    case = PagedCase(lens=lens, new=new, Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=torch.bfloat16, seed=D + 2)
    scale = 0.7 / math.sqrt(D)
    want = case.plain(scale, window)
    # a workgroup's form, row blocks x wavefronts that share out a row block's keys; 0: the kernel's own choice
    for form in [0, 41] + ([22] if D <= 128 else []) + ([42, 14] if D <= 64 else []):
        out = torch.full_like(case.qcat, float("nan"))
        ops.attention_prefill(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, 0, len(lens), max(new), Hq,
                              scale, window, out, form=form)
        got = out.double().cpu().numpy()
        assert np.isfinite(got).all(), form
        assert np.abs(got - want).max() < ATT_TOL[torch.bfloat16], form
    if D > 64:
        with pytest.raises(ops.KernelError, match="form 14"):
            ops.attention_prefill(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, 0, len(lens), max(new), Hq,
                                  scale, window, out, form=14)


@pytest.mark.parametrize("lens,new", [helpers.quick([64, 37, 1], [64, 37, 1]), ([64, 33], [2, 32]), helpers.quick([65, 20], [20, 20]), ([768, 5], [32, 5]),
                                      ([769, 64], [32, 32]), ([769, 64], [33, 64])])
def test_attention_prefill_of_short_portions_by_their_keys(ops, lens, new):
    """The kernel's own choice for up to 64 rows, at the lines between its forms: one tile of keys, up to and above 768."""
    case = PagedCase(lens=lens, new=new, Hq=3, Hkv=1, D=64, page=16, dtype=torch.bfloat16, seed=sum(lens))
    out = torch.full_like(case.qcat, float("nan"))
    ops.attention_prefill(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, 0, len(lens), max(new), 3, 0.1, None, out)
    assert np.abs(out.double().cpu().numpy() - case.plain(0.1, None)).max() < ATT_TOL[torch.bfloat16]


@pytest.mark.parametrize("lens,new", [([384, 9], [32, 9]), ([385, 30], [32, 2]), helpers.quick([400, 40], [3, 20]), ([700, 400], [16, 16])])
def test_attention_prefill_of_short_portions_of_small_heads(ops, lens, new):
    """Likewise at head size 32, whose line lies lower: more than 384 keys have the bits of 1 x 4, fewer those of 2 x 2."""
    case = PagedCase(lens=lens, new=new, Hq=2, Hkv=1, D=32, page=16, dtype=torch.bfloat16, seed=sum(lens))
    outs = [ops.attention_prefill(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, 0, len(lens), max(new), 2, 0.1, None,
                                  torch.full_like(case.qcat, float("nan")), form=f) for f in (0, 14 if max(lens) > 384 else 22)]
    assert np.abs(outs[0].double().cpu().numpy() - case.plain(0.1, None)).max() < ATT_TOL[torch.bfloat16]
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("Hq,Hkv,page,window,new", [
    helpers.quick(2, 1, 16, None, (1, 1, 1, 2)), (16, 16, 16, None, (1,) * 20 + (260, 129, 3)), (5, 5, 8, 100, (1, 1, 128)),
    (12, 4, 64, None, (1, 33, 64, 65)), helpers.quick(3, 3, 32, 40, (1, 1, 70)), (30, 30, 16, None, (1,) * 9 + (512, 40))])
def test_attention_of_one_token_sequences_and_portions_in_one_launch(ops, Hq, Hkv, page, window, new):
    """Few and many pairs, portions of 2 to 512 rows after nothing and after a past; the portions' rows have the bits of the prefill
    kernel's form of 4 row blocks x 2 key phases."""
    new = sorted(new, key=lambda n: n != 1)
    lens = [n + (37 * i * i) % 300 for i, n in enumerate(new)]
    nd = sum(n == 1 for n in new)
    case = PagedCase(lens=lens, new=new, Hq=Hq, Hkv=Hkv, D=64, page=page, dtype=torch.bfloat16, seed=Hq + page)
    assert ops._lib().da_attn_both_takes(nd, len(new) - nd, max(new), Hq, 64, page, 1)
    out = torch.full_like(case.qcat, float("nan"))
    ops.attention_both(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, nd, len(new) - nd, max(new), Hq, 0.09, window, out)
    assert np.abs(out.double().cpu().numpy() - case.plain(0.09, window)).max() < ATT_TOL[torch.bfloat16]
    alone = torch.full_like(case.qcat, float("nan"))
    ops.attention_prefill(case.qcat, case.cache, case.bt, case.q_start, case.seq_lens, nd, len(new) - nd, max(new), Hq, 0.09, window, alone, form=42)
    assert torch.equal(out[nd:], alone[nd:])


def test_when_attention_goes_in_one_launch(ops):
    takes = ops._lib().da_attn_both_takes
    assert takes(40, 1, 512, 16, 64, 16, 1) and takes(1, 1, 2, 12, 64, 16, 1)
    for a in ((0, 1, 512, 16, 64, 16, 1), (4, 0, 1, 16, 64, 16, 1), (4, 1, 512, 16, 48, 16, 1), (4, 1, 512, 16, 64, 16, 2), (4, 8, 1024, 16, 64, 16, 1),
              (4, 1, 512, 16, 64, 128, 1)):
        assert not takes(*a), a


def test_when_one_launch_is_ahead_of_two(ops):
    """The rule's lines: pairs of one-token rows, few rows beside them, keys in front of a short portion; never what the kernel
    does not take."""
    pays = ops._lib().da_attn_both_pays
    for a in ((40, 1, 512, 16, 64, 16, 1, 38), (64, 1, 2, 16, 64, 16, 1, 96), (100, 1, 16, 16, 64, 16, 1, 96), (63, 1, 512, 25, 64, 16, 1, 200), (1, 1, 65, 12, 64, 16, 1, 500), (30, 1, 64, 12, 64, 16, 1, 120)):
        assert pays(*a), a
    for a in ((65, 1, 15, 16, 64, 16, 1, 38), (65, 1, 16, 16, 64, 16, 1, 16), (128, 4, 512, 12, 64, 16, 1, 38), (101, 1, 512, 16, 64, 16, 1, 38), (255, 1, 64, 12, 64, 16, 1, 38), (30, 1, 64, 12, 64, 16, 1, 121), (30, 8, 2, 12, 64, 64, 1, 31),
              (0, 1, 512, 16, 64, 16, 1, 38), (4, 1, 512, 16, 48, 16, 1, 38), (4, 1, 512, 16, 64, 16, 2, 38)):
        assert not pays(*a), a


@pytest.mark.simt_quick
@pytest.mark.parametrize("form", [41, 42, 22, 14])
def test_attention_prefill_finds_a_far_key_in_every_phase(ops, form):
    """One key among 700 is made to stand out for one query row (key and query scaled up along one
    direction): the row's output is then that key's value, whichever wavefront's share the key lies in
    (with 2 or 4 wavefronts to a row block a share is every 2nd or 4th tile of 64 keys) and wherever
    in its tile."""
    Hq, Hkv, D, page, n = 2, 2, 64, 16, 700
    case = PagedCase(lens=[n], new=[n], Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=torch.bfloat16, seed=31)
    scale = 1.0 / math.sqrt(D)
    row = n - 1
    for far in (0, 63, 64, 129, 200, 300, 447, 640, 699):
        q = case.qcat.clone()
        cache = case.cache.clone()
        pg, r = int(case.bt[0, far // page]), far % page
        direction = torch.zeros(D); direction[far % D] = 30.0
        for h in range(Hq):
            q[row, h * D:(h + 1) * D] = direction.to(torch.bfloat16)
            cache[pg, 0, h, r, :] = direction.to(torch.bfloat16)
        out = torch.empty_like(q)
        ops.attention_prefill(q, cache, case.bt, case.q_start, case.seq_lens, 0, 1, n, Hq, scale, None, out, form=form)
        for h in range(Hq):
            value = cache[pg, 1, h].reshape(D, page)[:, r].float()          # values lie dimension-major in a page
            assert (out[row, h * D:(h + 1) * D].float() - value).abs().max() < 2e-2, (far, h)


@pytest.mark.simt_quick
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_row_that_sees_no_key_gives_zeros(ops, dtype):
    """The padding rows of a fixed-shape decode step: length 0, a block table of -1.  Zeros, never NaN
    (NaN would spread through the row's residual into its logits and into the sampling kernel)."""
    Hq, Hkv, D, page = 4, 2, 32, 16
    case = PagedCase(lens=[20, 7], new=[1, 1], Hq=Hq, Hkv=Hkv, D=D, page=page, dtype=dtype, seed=8)
    q = torch.cat([case.qcat, torch.randn(2, Hq * D).to(dtype).to(DEV)])
    bt = torch.cat([case.bt, torch.full((2, case.bt.shape[1]), -1, dtype=torch.int32, device=DEV)])
    seq_of = torch.tensor([0, 1, 2, 3], dtype=torch.int32, device=DEV)
    pos = torch.tensor([19, 6, 0, 0], dtype=torch.int32, device=DEV)
    out = torch.full_like(q, float("nan"))
    ops.attention_ref(q, case.cache, bt, seq_of, pos, Hq, 0.2, None, out)
    want = case.plain(0.2, None)
    assert np.abs(out[:2].double().cpu().numpy() - want).max() < ATT_TOL[dtype]
    assert torch.equal(out[2:], torch.zeros_like(out[2:]))
    if dtype == torch.bfloat16:
        out2 = torch.full_like(q, float("nan"))
        lens = torch.tensor([20, 7, 0, 0], dtype=torch.int32, device=DEV)
        ops.attention_decode(q, case.cache, bt, lens, 4, Hq, 0.2, None, out2)
        assert torch.equal(out2[2:], torch.zeros_like(out2[2:]))
        assert np.abs(out2[:2].double().cpu().numpy() - want).max() < ATT_TOL[dtype]


@pytest.mark.simt_quick
def test_attention_reference_vector_shape(ops):
    """The shape of the reference's own paged-attention test: 4 query heads on 2 key heads, head 8
    there (16 here: head sizes come in steps of 16), pages of 3 rows there (16 here), 5 visible rows,
    scale 0.25, inputs by its closed formula (tensor/src/test/java/io/teknek/deliverance/tensor/
    operations/TensorOperationsDecodePagedAttentionTest.java:18-47,92-99)."""
    Hq, Hkv, D, page, rows = 4, 2, 16, 16, 5

    def tensor(r, c, seed):
        return torch.tensor([[(((i * 19 + j * 23 + seed) % 43) - 21) / 21.0 for j in range(c)] for i in range(r)])
    q = tensor(1, Hq * D, 3)
    k = torch.cat([tensor(3, Hkv * D, 7), tensor(3, Hkv * D, 11)])[:rows]
    v = torch.cat([tensor(3, Hkv * D, 13), tensor(3, Hkv * D, 17)])[:rows]
    want = P.causal_attention(q.double().numpy(), k.double().numpy(), v.double().numpy(), Hq, 0.25, n_kv_head=Hkv, past=rows - 1)
    for dtype in (torch.float32, torch.bfloat16):
        cache = torch.full((2, 2, Hkv, page, D), float("nan"), dtype=dtype, device=DEV)
        qkv = torch.cat([torch.zeros(rows, Hq * D), k, v], dim=1).to(dtype).to(DEV)
        slots = torch.tensor([16 + i for i in range(rows)], dtype=torch.int32, device=DEV)     # page 1
        ops.kv_write(qkv, Hq * D, Hq * D + Hkv * D, cache, slots, Hkv, D)
        bt = torch.tensor([[1]], dtype=torch.int32, device=DEV)
        qd = q.to(dtype).to(DEV)
        out = torch.empty_like(qd)
        ops.attention_ref(qd, cache, bt, torch.zeros(1, dtype=torch.int32, device=DEV),
                          torch.tensor([rows - 1], dtype=torch.int32, device=DEV), Hq, 0.25, None, out)
        tol = 1e-5 if dtype == torch.float32 else 2e-2
        assert np.abs(out.double().cpu().numpy() - want).max() < tol
        if dtype == torch.bfloat16:
            out2 = torch.empty_like(qd)
            ops.attention_decode(qd, cache, bt, torch.tensor([rows], dtype=torch.int32, device=DEV), 1, Hq, 0.25, None, out2)
            assert np.abs(out2.double().cpu().numpy() - want).max() < tol


@pytest.mark.simt_quick
@pytest.mark.parametrize("page", [16, 32, 64])
@pytest.mark.parametrize("N", [40, 600])
def test_cache_write_puts_every_key_and_value_in_its_row(ops, N, page):
    """Both write kernels (a token a workgroup; 16 tokens a workgroup from 256 tokens on) against
    direct placement: whole aligned pages in order, runs that start inside a page, single rows
    all over, and tokens whose keys are not kept (-1)."""
    Hq, Hkv, D = 3, 2, 48
    g = torch.Generator().manual_seed(N + page)
    n_pages = 4 * (N // page + 2)
    free = torch.randperm(n_pages, generator=g).tolist()
    slots = []
    while len(slots) < N:
        kind = len(slots) // 16 % 4
        pg = free.pop()
        if kind == 0:      # a whole page in order
            slots += [pg * page + i for i in range(page)]
        elif kind == 1:    # a run that starts inside the page
            slots += [pg * page + i for i in range(5, page)]
        elif kind == 2:    # rows of a page in any order
            slots += [pg * page + int(i) for i in torch.randperm(page, generator=g)[:11]]
        else:              # not kept
            slots += [-1] * 7
    slots = slots[:N]
    qkv = bf(torch.randn(N, (Hq + 2 * Hkv) * D, generator=g)).to(DEV)
    st = torch.tensor(slots, dtype=torch.int32, device=DEV)
    for dtype in (torch.bfloat16, torch.float32):
        x = qkv.to(dtype)
        cache = torch.zeros(n_pages, 2, Hkv, page, D, dtype=dtype, device=DEV)
        ops.kv_write(x, Hq * D, (Hq + Hkv) * D, cache, st, Hkv, D)
        want = torch.zeros(n_pages, 2, Hkv, page, D, dtype=dtype)
        want_v = torch.zeros(n_pages, Hkv, D, page, dtype=dtype)          # values lie dimension-major in a page
        xc = x.cpu()
        for n, sl in enumerate(slots):
            if sl < 0:
                continue
            pg, row = divmod(sl, page)
            want[pg, 0, :, row, :] = xc[n, Hq * D:(Hq + Hkv) * D].view(Hkv, D)
            want_v[pg, :, :, row] = xc[n, (Hq + Hkv) * D:].view(Hkv, D)
        got = cache.cpu()
        assert torch.equal(got[:, 0], want[:, 0])
        assert torch.equal(got[:, 1].reshape(n_pages, Hkv, D, page), want_v)


def test_a_far_key_among_hundreds_is_found(ops):
    """Random keys give near-uniform weights, which would hide a lost key: here one key far back
    carries almost all the weight of the last query."""
    for far, n in ((3, 700), (255, 700), (256, 700), (639, 700)):
        case = PagedCase(lens=[n], new=[1], Hq=2, Hkv=2, D=64, page=16, dtype=torch.bfloat16, seed=far, scale_boost=(far, 3.0))
        scale = 1 / 8
        want = case.plain(scale, None)
        # the weight of the far key dominates: the result is close to that key's value
        assert np.abs(want[0, :64] - case.v[0][far, :64].double().numpy()).max() < 0.2
        out = torch.empty_like(case.qcat)
        ops.attention_decode(case.qcat, case.cache, case.bt, case.seq_lens, 1, 2, scale, None, out)
        assert np.abs(out.double().cpu().numpy() - want).max() < 2e-2
        case2 = PagedCase(lens=[n], new=[130], Hq=2, Hkv=2, D=64, page=16, dtype=torch.bfloat16, seed=far, scale_boost=(far, 3.0))
        out2 = torch.empty_like(case2.qcat)
        ops.attention_prefill(case2.qcat, case2.cache, case2.bt, case2.q_start, case2.seq_lens, 0, 1, 130, 2, scale, None, out2)
        assert np.abs(out2.double().cpu().numpy() - case2.plain(scale, None)).max() < 2e-2


# ----------------------------------------------------------------------------- sampling
def _records(params_list, V, seeds):
    import struct
    from deliverance_amd.sampling import JavaRandom, device_record
    words, us = [], []
    for p, seed in zip(params_list, seeds):
        rng = JavaRandom(seed)
        rec = device_record(p, rng, V)
        words += struct.unpack("<8i", rec)
        us.append(struct.unpack("<fififfii", rec)[4])
    return torch.tensor(words, dtype=torch.int32, device=DEV), us


def test_sampling_kernel_against_the_plain_sampler(ops):
    from deliverance_amd.sampling import GeneratorParameters as GP
    g = torch.Generator().manual_seed(5)
    V = 50257
    combos = [GP(), GP(temperature=0.8), GP(temperature=1.3, top_k=50), GP(temperature=0.7, top_p=0.9),
              GP(temperature=1.0, top_k=40, top_p=0.95), GP(temperature=1.0, top_k=0.999), GP(temperature=2.0, top_p=0.3),
              GP(temperature=0.9, top_k=5, top_p=0.5, uniform_top_p=1.0), GP(temperature=1.0, top_p=1.0)]
    rows, plist, seeds = [], [], []
    for i in range(4):
        for c in combos:
            rows.append(torch.randn(V, generator=g) * 3.0)
            plist.append(c); seeds.append(100 + i)
    logits = torch.stack(rows).to(DEV)
    rec, us = _records(plist, V, seeds)
    out = torch.empty(len(rows), dtype=torch.int32, device=DEV)
    ops.sample(logits, rec, out)
    got = out.cpu().tolist()
    for r, (p, u) in enumerate(zip(plist, us)):
        lg = rows[r].numpy()
        want = int(np.argmax(lg)) if p.temperature == 0 else \
            P.sample_top_k_top_p(lg, p.temperature, p.top_k, p.top_p, p.uniform_top_p, u)
        assert got[r] == want, (r, p)


@pytest.mark.simt_quick
def test_sampling_vectors_of_the_reference(ops):
    """core/src/test/java/io/teknek/deliverance/model/TopKSamplerTest.java:23-54, with the draws given."""
    import struct
    logits = torch.tensor([[5.0, 4.0, 3.0, 2.0, 1.0]] * 5 + [[1.0, 1.0, 1.0, 0.0, 1.0]] * 2, device=DEV)

    def rec(T, k, p, uni, u):
        return struct.unpack("<8i", struct.pack("<fififfii", T, k, p, uni, u, 0.0, 0, 0))
    words = (rec(1.0, 2, 0.95, 0, 0.99) + rec(1.0, 2, 0.95, 0, 0.60) + rec(1.0, 2, 0.95, 1, 0.60) + rec(0.0, 0, 0.0, 0, 0.0)
             + rec(1.0, 0, 0.0, 0, 0.999999) + rec(0.0, 0, 0.0, 0, 0.0) + rec(1.0, 3, 0.0, 0, 0.70))
    out = torch.empty(7, dtype=torch.int32, device=DEV)
    ops.sample(logits, torch.tensor(words, dtype=torch.int32, device=DEV), out)
    # weighted 0.99 -> 1, weighted 0.60 -> 0, uniform in nucleus 0.60 -> 1, greedy -> 0, u ~ 1 -> last token,
    # greedy ties -> lowest index, top-3 of equal logits keeps indices 0,1,2 and 0.70 lands on the third
    assert out.cpu().tolist() == [1, 0, 1, 0, 4, 0, 2]


@pytest.mark.simt_quick
def test_xtc_and_logprobs(ops):
    import struct
    V = 1000
    g = torch.Generator().manual_seed(9)
    lg = torch.randn(V, generator=g)
    lg[10], lg[20], lg[30] = 9.0, 8.5, 8.0          # three tokens above a 10% threshold
    logits = torch.stack([lg, lg, lg]).to(DEV)

    def rec(T, thr, active):
        return struct.unpack("<8i", struct.pack("<fififfii", T, 0, 0.0, 0, 0.0, thr, active, 0))
    words = rec(0.0, 0.1, 1) + rec(0.0, 0.1, 0) + rec(1.0, 0.1, 1)
    out = torch.empty(3, dtype=torch.int32, device=DEV)
    params = torch.tensor(words, dtype=torch.int32, device=DEV)
    ops.sample(logits, params, out)
    # active: the least likely of the tokens above the threshold; inactive: the maximum
    assert out.cpu().tolist() == [30, 10, 30]
    idx = torch.empty(3, 4, dtype=torch.int32, device=DEV)
    lp = torch.empty(3, 4, dtype=torch.float32, device=DEV)
    ops.top_logprobs(logits, params, 4, idx, lp)
    want = torch.log_softmax(lg.double(), 0)
    top = torch.topk(want, 4)
    assert idx[0].cpu().tolist() == top.indices.tolist()
    assert (lp[0].cpu().double() - top.values).abs().max() < 1e-4


# ----------------------------------------------------------------------------- fused norm + product
@pytest.mark.parametrize("M,N,K", [helpers.quick(1, 96, 64), (8, 2304, 768), helpers.quick(17, 1000, 96), (32, 200, 1600), (5, 50257, 768),
                                   (16, 520, 1024), helpers.quick(12, 72, 1000), helpers.quick(9, 40, 520), (3, 1000, 1600), (16, 300, 2048),
                                   helpers.quick(5, 64, 1304), helpers.quick(2, 48, 8), (11, 200, 1992), (8, 200, 1280),
                                   helpers.quick(7, 48, 2040)])
@pytest.mark.parametrize("pdtype", [torch.bfloat16, torch.float32])
def test_fused_norm_product(ops, M, N, K, pdtype):
    helpers.skip_in_simulation_if(M * N * K > 1.2e8)
    g = torch.Generator().manual_seed(M + N)
    x = (torch.randn(M + 3, K, generator=g) * 2 + 1).to(DEV)
    gw, gb = torch.randn(K, generator=g).to(pdtype).to(DEV), torch.randn(K, generator=g).to(pdtype).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    # the product's bias in the norm's dtype (the kernels for parameters of one dtype) or, with 32-bit norm
    # parameters and an even M, in bfloat16 (the general kernel)
    bias = bf(torch.randn(N, generator=g)).to(pdtype if M % 2 else torch.bfloat16).to(DEV)
    rows = torch.tensor([(i * 7) % (M + 3) for i in range(M)], dtype=torch.int32, device=DEV)
    a = F.layer_norm(x.double(), (K,), gw.double(), gb.double(), 1e-5)[rows.long()].to(torch.bfloat16).double()
    for act, od in ((None, torch.float32), ("gelu_new", torch.bfloat16)):
        out = torch.empty(M, N, device=DEV, dtype=od)
        ops.linear_ln(x, rows, M, gw, gb, 1e-5, w, bias, out, act=act)
        ref = a @ w.double().t() + bias.double()
        if act:
            ref = F.gelu(ref, approximate="tanh")
        tol = (2e-2 if od == torch.bfloat16 else 2e-3) * max(1.0, ref.abs().max().item())
        assert (out.double() - ref).abs().max() < tol


@pytest.mark.parametrize("M", [helpers.quick(5), helpers.quick(40), helpers.quick(300), 1000, 2100])
def test_product_writes_keys_and_values(ops, M):
    """The skinny (M <= 64) and tile kernels scatter the k | v columns in their epilogue."""
    g = torch.Generator().manual_seed(M)
    Hq, Hkv, D, page, K = 5, 3, 48, 16, (128 if M >= 2000 else 104)      # a K that no slab cuts, too
    N = (Hq + 2 * Hkv) * D
    n_pages = (M + page - 1) // page + 2
    a = bf(torch.randn(M, K, generator=g)).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    bias = bf(torch.randn(N, generator=g)).to(DEV)
    perm = torch.randperm(n_pages * page, generator=g)[:M].to(torch.int32)
    perm[M // 2] = -1
    # the places in any order; and as a prompt portion has them: runs of consecutive rows, one from a
    # multiple of 8 on (values go over in 16-byte runs), one from 3 on, with a token that is not kept
    runs = torch.cat([torch.arange(16, 16 + M // 2), torch.arange(16 + M // 2 + 19, 16 + M // 2 + 19 + M - M // 2)]).to(torch.int32)
    runs[M // 4] = -1
    for order in (perm, runs):
        slots = order.to(DEV)
        c1 = torch.zeros(n_pages + 2, 2, Hkv, page, D, dtype=torch.bfloat16, device=DEV)
        c2 = torch.zeros_like(c1)
        out1 = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        out2 = torch.empty_like(out1)
        ops.linear_mfma(a, w, bias, out1, kv_cache=c1, slot_map=slots, q_cols=Hq * D)
        ops.linear_mfma(a, w, bias, out2)
        ops.kv_write(out2, Hq * D, (Hq + Hkv) * D, c2, slots, Hkv, D)
        assert torch.equal(out1, out2)
        assert torch.equal(c1, c2) and c1.abs().sum() > 0


@pytest.mark.parametrize("M,K,Dv,N", [helpers.quick(17, 72, 16, 4160), helpers.quick(5, 1288, 24, 4160), (5, 1288, 16, 5120), (17, 72, 24, 8192),
                                      (33, 136, 16, 4801), (64, 72, 24, 8192), (64, 136, 16, 4100), (3, 72, 24, 4160), (9, 72, 16, 1000), (40, 72, 24, 900)])
def test_split_product_keeps_no_column_behind_the_values(ops, M, K, Dv, N):
    """q | k | v | rest: keys and values of the rows with a place are in it, bit for bit the product's columns, and every other
    entry of the cache is what it was; one workgroup a compute unit (4,097 to 8,192 columns) and the other forms for few rows."""
    g = torch.Generator().manual_seed(M + N)
    Hkv, D, page, P, rest = 2, 16, 16, 6, 100
    q_cols = N - rest - Hkv * (D + Dv)
    a, w, bias = (bf(torch.randn(*shape, generator=g)).to(DEV) for shape in ((M, K), (N, K), (N,)))
    slots = torch.randperm((P - 1) * page, generator=g)[:M].to(torch.int32)
    slots[M // 2] = -1
    slots[0] = (P - 2) * page + 3 if not bool((slots == (P - 2) * page + 3).any()) else slots[0]
    cache = bf(torch.randn(P, Hkv * page * (D + Dv), generator=g)).to(DEV)
    want = cache.cpu().clone()
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    ops.linear_kv_split(a, w, bias, out, cache, slots.to(DEV), q_cols, Hkv, D, Dv, page)
    ref = a.double().cpu() @ w.double().cpu().t() + bias.double().cpu()
    assert (out.double().cpu() - ref).abs().max() <= 2.0 ** -8 * ref.abs().max() + 1e-3
    for m, slot in enumerate(slots.tolist()):
        if slot < 0:
            continue
        pg, row = divmod(slot, page)
        kv = out[m, q_cols:].cpu()
        want[pg, :Hkv * page * D].view(Hkv, page, D)[:, row] = kv[:Hkv * D].view(Hkv, D)
        want[pg, Hkv * page * D:].view(Hkv, Dv, page)[:, :, row] = kv[Hkv * D:Hkv * (D + Dv)].view(Hkv, Dv)
    assert torch.equal(cache.cpu(), want)


@pytest.mark.simt_quick
@pytest.mark.parametrize("M,K", [(9, 96), (7, 1312)])
def test_fused_norm_product_writes_keys_and_values(ops, M, K):
    """(7 rows and a wide K: two groups of 16 columns a workgroup)"""
    g = torch.Generator().manual_seed(11)
    Hq, Hkv, D, page = 6, 2, 48, 16
    N = (Hq + 2 * Hkv) * D
    x = torch.randn(M, K, generator=g).to(DEV)
    gw, gb = bf(torch.randn(K, generator=g)).to(DEV), bf(torch.randn(K, generator=g)).to(DEV)
    w = bf(torch.randn(N, K, generator=g) * 0.1).to(DEV)
    bias = bf(torch.randn(N, generator=g)).to(DEV)
    slots = torch.tensor([3 * page + 5, -1, 0, 17, 40, 41, 42, 95, 64][:M], dtype=torch.int32, device=DEV)
    c1 = torch.zeros(6, 2, Hkv, page, D, dtype=torch.bfloat16, device=DEV)
    c2 = torch.zeros_like(c1)
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    ops.linear_ln(x, None, M, gw, gb, 1e-5, w, bias, out, kv_cache=c1, slot_map=slots, q_cols=Hq * D)
    ops.kv_write(out, Hq * D, (Hq + Hkv) * D, c2, slots, Hkv, D)      # the separate kernel on the same rows
    assert torch.equal(c1, c2) and c1.abs().sum() > 0


@pytest.mark.parametrize("form", ["decode", "split", "gated", "split gated", "prefill", "32-bit"])
def test_attention_of_more_sequences_than_a_launch_has_rows(ops, form):
    """65,600 sequences of one token with 1, 2, 66 or 67 keys: a launch's second size ends at 65,535, so the last ones go in another,
    with their rows of q, table, gate, result and of the shares' sums."""
    helpers.skip_in_simulation_if(True)
    g = torch.Generator().manual_seed(3)
    dtype = torch.float32 if form == "32-bit" else torch.bfloat16
    S, Hq, D, page, P, B = 65600, 2, 16, 16, 9, 8
    cache = torch.randn(P, 2, Hq, page * D, generator=g).to(dtype).to(DEV)
    q = torch.randn(S, Hq * D, generator=g).to(dtype).to(DEV)
    gate = torch.randn(S, Hq * D, generator=g).to(dtype).to(DEV)
    table = torch.randint(0, P, (S, B), generator=g, dtype=torch.int32).to(DEV)
    lens = torch.tensor([1, 2, 66, 67], dtype=torch.int32)[torch.randint(0, 4, (S,), generator=g)].to(DEV)
    starts = torch.arange(S + 1, dtype=torch.int32, device=DEV)
    out = torch.zeros(S, Hq * D, dtype=dtype, device=DEV)
    n = 2 if "split" in form else 1
    shares = torch.empty(S * Hq * n * (D + 2), device=DEV)
    lib, stream = ops._lib(), ops._stream()
    rows = (q.data_ptr(), Hq * D, cache.data_ptr(), table.data_ptr(), B)
    sizes, result = (Hq, Hq, D, page, 0.25, 0), (out.data_ptr(), Hq * D)
    if form == "decode":
        rc = lib.da_attn_decode(*rows, lens.data_ptr(), S, *sizes, *result, stream)
    elif form == "split":
        rc = lib.da_attn_decode_split(*rows, lens.data_ptr(), S, *sizes, *result, n, shares.data_ptr(), shares.numel() * 4, stream)
    elif "gated" in form:
        rc = lib.da_attn_decode_rel(*rows, lens.data_ptr(), S, *sizes, None, 0, None, 0.0, 0, 0, None, gate.data_ptr(), Hq * D, *result, n,
                                    shares.data_ptr(), shares.numel() * 4, stream)
    elif form == "prefill":
        rc = lib.da_attn_prefill(*rows, starts.data_ptr(), lens.data_ptr(), 0, S, 1, *sizes, *result, 0, stream)
    else:
        rc = lib.da_attn_f32(*rows, starts.data_ptr(), lens.data_ptr(), S, 1, *sizes, *result, stream)
    assert rc == 0
    at = torch.tensor([0, 1, 32799, 32800, 65534, 65535, 65536, S - 1])
    pages = cache.double().cpu()[table.cpu()[at].long()]                                # [8, B, 2, Hq, page * D]
    k = pages[:, :, 0].reshape(-1, B, Hq, page, D).transpose(1, 2).reshape(-1, Hq, B * page, D)
    v = pages[:, :, 1].reshape(-1, B, Hq, D, page).permute(0, 2, 1, 4, 3).reshape(-1, Hq, B * page, D)
    score = (q.double().cpu()[at].reshape(-1, Hq, 1, D) * k).sum(-1) * 0.25
    score = score.masked_fill(torch.arange(B * page)[None, None] >= lens.cpu()[at].long()[:, None, None], -float("inf"))
    want = (score.softmax(-1)[..., None] * v).sum(2).reshape(-1, Hq * D)
    if "gated" in form:
        want = want * torch.sigmoid(gate.double().cpu()[at])
    tol = 2.0 ** -8 * want.abs() + 1e-4 if dtype == torch.bfloat16 else torch.full_like(want, 1e-5)
    if form == "prefill":
        tol = tol + 2.0 ** -8 * v.abs().max()                                           # (its weights are bfloat16)
    assert ((out.double().cpu()[at] - want).abs() <= tol).all()
    assert bool((out != 0).any(dim=1).all())


@pytest.mark.parametrize("window", [None, 100])
def test_prefill_attention_has_the_same_bits_wherever_q_is_asked_for(ops, window):
    """Head size 64 without phases: a launch of more than 640 workgroups asks for q first, its halves behind the first tile (attn_prefill.hip); portions
    that end inside a row block, tiles that a window or the length cuts, a sequence with no rows."""
    helpers.skip_in_simulation_if(True)
    g = torch.Generator().manual_seed(5)
    n, H, page = 24, 16, 16
    new = [0 if i == 7 else 130 + 9 * i for i in range(n)]
    lens = [t + 13 * (i % 5) for i, t in enumerate(new)]
    pages = [-(-max(1, l) // page) for l in lens]
    bt = torch.zeros(n, max(pages), dtype=torch.int32)
    for i, p in enumerate(pages):
        bt[i, :p] = torch.arange(sum(pages[:i]), sum(pages[:i + 1]))
    cache = bf(torch.randn(sum(pages), 2, H, page, 64, generator=g)).to(DEV)
    at = [sum(new[:i]) for i in range(n + 1)]
    q = bf(torch.randn(at[-1], H * 64, generator=g)).to(DEV)
    bt, starts, sl = bt.to(DEV), torch.tensor(at, dtype=torch.int32, device=DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)
    run = lambda s0, m, out: ops.attention_prefill(q, cache, bt, starts, sl, s0, m, max(new), H, 0.125, window, out, form=41)
    assert H * n * -(-max(new) // 128) > 640 >= H * (n // 2) * -(-max(new) // 128)
    whole = run(0, n, torch.zeros(at[-1], H * 64, dtype=torch.bfloat16, device=DEV))
    halves = run(n // 2, n // 2, run(0, n // 2, torch.zeros_like(whole)))
    assert torch.equal(whole, halves) and bool((whole != 0).any(dim=1).all())


@pytest.mark.parametrize("K,F", [helpers.quick(72, 24), (128, 40), (136, 20), (1024, 344), (1376, 72), (1544, 36)])
@pytest.mark.parametrize("gated", [True, False])
def test_grouped_products_of_experts_with_few_rows(ops, K, F, gated):
    """Tiles of 32 slots whose filled slots are 1 to 32 (both sides of 8, 16, and whole loads of 8 rows), an expert with two tiles, a tile of nobody;
    columns that end inside a workgroup, a K that a step cuts, two and three steps a wavefront; slots without a pair are not written.  First
    products gathered by slot with a weight a slot (one matrix) or gate and up (two), the second on the slots' own rows.  Bounds: 2^-8 of the
    largest entry for the bfloat16 results, 1e-5 of it for the 32-bit sums."""
    g = torch.Generator().manual_seed(K + F)
    counts, tile = [1, 8, 9, 16, 17, 24, 25, 32 + 5], 32
    E, N = len(counts), 41
    rows, experts = [], []
    for e, c in enumerate(counts):
        for t0 in range(0, c, tile):
            n = min(tile, c - t0)
            rows += [int(x) for x in torch.randint(0, N, (n,), generator=g)] + [-1] * (tile - n)
            experts.append(e)
    rows, experts = rows + [-1] * tile, experts + [-1]
    T = len(experts)
    row_of_slot, tile_expert = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in (rows, experts))
    G = 2 if gated else 1
    h = bf(torch.randn(N, K, generator=g)).to(DEV)
    up = bf(torch.randn(E, G * F, K, generator=g) * 0.1).to(DEV)
    scale = torch.rand(T * tile, generator=g).to(DEV) + 0.5
    mid = torch.full((T * tile, F), 7.0, dtype=torch.bfloat16, device=DEV)
    lib, ptr = ops._lib(), ops._ptr
    if gated:
        ops._check(lib.da_moe_gated_mfma(ptr(h), K, ptr(row_of_slot), ptr(tile_expert), ptr(up), ptr(mid), F, T, K, F, ops.ACTIVATIONS["silu"],
                                         0.0, ops._stream()))
    else:
        ops._check(lib.da_moe_up_mfma(ptr(h), K, ptr(row_of_slot), ptr(tile_expert), ptr(up), ptr(scale), ptr(mid), F, T, K, F,
                                      ops.ACTIVATIONS["relu"], ops._stream()))
    used = row_of_slot >= 0
    expert_of = tile_expert.long().repeat_interleave(tile)
    hd, ud = h.double(), up.double()
    for e in range(E):
        at = (used & (expert_of == e)).nonzero()[:, 0]
        first = hd[row_of_slot[at].long()] @ ud[e].t()
        want = F_silu(first[:, :F]) * first[:, F:] if gated else F_relu(first * scale[at].double()[:, None])
        assert (mid[at].double() - want).abs().max() < 2.0 ** -8 * max(1.0, want.abs().max().item()), (e, counts[e])
    assert bool((mid[~used] == 7.0).all())
    if F % 8:
        return                                       # (rows of the second product's operands are whole pieces of 16 bytes)
    down = bf(torch.randn(E, K, F, generator=g) * 0.1).to(DEV)
    out = torch.full((T * tile, K), 7.0, device=DEV)
    ops._check(lib.da_moe_down_mfma(ptr(mid), F, ptr(row_of_slot), ptr(tile_expert), ptr(down), ptr(out), K, T, F, K, ops._stream()))
    for e in range(E):
        at = (used & (expert_of == e)).nonzero()[:, 0]
        want = mid[at].double() @ down[e].double().t()
        assert (out[at].double() - want).abs().max() < 1e-5 * max(1.0, want.abs().max().item()), (e, counts[e])
    assert bool((out[~used] == 7.0).all())


def F_silu(x):
    return x / (1.0 + torch.exp(-x))


def F_relu(x):
    return x.clamp(min=0.0)
