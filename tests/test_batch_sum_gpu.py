"""Products summed over the batch (cpmk_gemm_int8_scale_sum, cpmk_gemm_fp16_sum) against float64, at the sizes where their
tiles, slabs and groups change."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck

pytestmark = pytest.mark.gpu

# batch, groups, n, m, k: one entry; partial tiles; one slab per entry; several groups; 16 entries; 256x128 tiles (the last three)
SHAPES = [(1, 1, 4, 4, 128), (3, 1, 132, 260, 128), (4, 2, 128, 128, 256), (16, 1, 36, 200, 384), (6, 3, 300, 124, 640),
          (2, 1, 4100, 2052, 128), (5, 1, 3080, 3072, 256), (8, 4, 1024, 1028, 512)]


def _st():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("shape", SHAPES)
def test_int8_sum(gpu, shape):
    batch, groups, n, m, k = shape
    print("int8 sum", shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)
    A = torch.randint(-128, 128, (batch, m, k), generator=g, device="cuda", dtype=torch.int8)
    B = torch.randint(-128, 128, (batch, n, k), generator=g, device="cuda", dtype=torch.int8)
    s = (torch.rand((batch, n), generator=g, device="cuda") * 1e-3 + 1e-4).half()
    out = torch.full((groups, n, m), float("nan"), device="cuda", dtype=torch.half)
    ck.gemm_int8_scale_sum(m, k, n, batch, groups, A.data_ptr(), B.data_ptr(), s.data_ptr(), out.data_ptr(), _st())
    for q in range(groups):
        want = torch.zeros((n, m), device="cuda", dtype=torch.float64)
        mag = torch.zeros_like(want)
        for e in range(q * batch // groups, (q + 1) * batch // groups):
            acc = (B[e].double() @ A[e].double().t()) * s[e].double()[:, None]      # exact integers (|acc| < 2^53) times the scale
            want += acc
            mag += acc.abs()
        # one fp32 rounding per entry (the fused multiply-add) and one of the conversion of a 24-bit integer, then one to fp16
        bound = mag * (batch + 1) * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25
        assert bool(((out[q].double() - want).abs() <= bound).all()), shape


@pytest.mark.parametrize("k", [34, 64, 66, 72, 96, 128, 320, 500])
@pytest.mark.parametrize("shape", [(1, 1, 4, 4), (4, 2, 132, 260), (3, 1, 128, 512), (2, 1, 3588, 3584)])
def test_fp16_sum(gpu, shape, k):
    batch, groups, n, m = shape
    print("fp16 sum", shape, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)
    A = torch.randn((batch, m, k), generator=g, device="cuda").half()
    B = torch.randn((batch, n, k), generator=g, device="cuda").half()
    out = torch.full((groups, n, m), float("nan"), device="cuda", dtype=torch.half)
    ck.gemm_fp16_sum(m, k, n, batch, groups, A.data_ptr(), B.data_ptr(), out.data_ptr(), _st())
    per = batch // groups
    for q in range(groups):
        want = torch.zeros((n, m), device="cuda", dtype=torch.float64)
        mag = torch.zeros_like(want)
        for e in range(q * per, (q + 1) * per):
            want += B[e].double() @ A[e].double().t()
            mag += B[e].double().abs() @ A[e].double().abs().t()
        bound = mag * (per * k) * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25      # fp32 sums in any order, one rounding to fp16
        assert bool(((out[q].double() - want).abs() <= bound).all()), (shape, k)


def test_groups(gpu):
    for m, n, batch in ((4, 4, 1), (512, 512, 8), (4096, 10240, 8), (4096, 4096, 13), (64, 64, 7), (8192, 8192, 64)):
        groups = ck.gemm_sum_groups(m, n, batch)
        assert 1 <= groups <= batch and batch % groups == 0 and (groups == batch or batch // groups <= 16)


def test_groups_fill_the_device(gpu):
    """No sum over the batch whose last round of tiles leaves the device mostly idle."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for m, n, batch in ((896, 5376, 16), (5376, 3328, 12), (4096, 4352, 8), (4096, 4096, 8), (2560, 2560, 5), (1536, 1536, 12)):
        for kind in (1, 2):
            for k in (68, 128, 512):
                groups = ck.gemm_sum_groups_for(kind, m, k, n, batch)
                assert 1 <= groups <= batch and batch % groups == 0
                if groups < batch:
                    fit = [-(-n // t) * -(-m // t) * groups for t in (128, 256)]
                    fill = [t / cus / (t // cus + (0 if t % cus == 0 else 0.5 if 2 * (t % cus) <= cus else 1)) for t in fit]
                    assert max(fill) >= 0.75, (m, n, batch, kind, k, groups)


@pytest.mark.parametrize("kind", [0, 1, 2])       # int8, fp16 K-major, fp16 (K, rows)
@pytest.mark.parametrize("batch", [1, 2, 7, 12, 16, 17, 32, 34, 48, 1009])
def test_quickest_groups(gpu, kind, batch):
    """A divisor of the batch whose groups the sums take (16 entries; (K, rows), one contraction, operands below 4 GiB), or the batch: one by one."""
    for m, n in ((4, 4), (512, 512), (832, 1856), (1280, 3328), (2560, 2560), (8192, 8192)):
        for k in (40, 66, 128, 1000, 4096):
            groups = ck.gemm_sum_groups_timed(kind, m, k, n, batch)
            assert 1 <= groups <= batch and batch % groups == 0, (m, n, k, groups)
            if groups < batch:
                if kind == 2:
                    assert max(m, n) * k * (batch // groups) * 2 < 1 << 32, (m, n, k, groups)
                else:
                    assert batch // groups <= 16, (m, n, k, groups)


@pytest.mark.parametrize("shape", [s for s in SHAPES if s[1] > 1])
def test_int8_parts(gpu, shape):
    batch, groups, n, m, k = shape
    print("int8 parts", shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)
    A = torch.randint(-128, 128, (batch, m, k), generator=g, device="cuda", dtype=torch.int8)
    B = torch.randint(-128, 128, (batch, n, k), generator=g, device="cuda", dtype=torch.int8)
    s = (torch.rand((batch, n), generator=g, device="cuda") * 1e-1 + 1e-2).half()        # (sums beyond fp16's range among them)
    parts = torch.full((groups, n, m), float("nan"), device="cuda")
    ck.gemm_int8_scale_parts(m, k, n, batch, groups, A.data_ptr(), B.data_ptr(), s.data_ptr(), parts.data_ptr(), _st())
    acc = torch.stack([(B[e].double() @ A[e].double().t()) * s[e].double()[:, None] for e in range(batch)]).view(groups, -1, n, m)
    bound = acc.abs().sum(1) * (batch + 1) * 2.0 ** -24        # a rounding per entry and one of a 24-bit integer's conversion
    assert bool(((parts.double() - acc.sum(1)).abs() <= bound).all()), shape
    _check_add(parts)


@pytest.mark.parametrize("k_first,k", [(False, k) for k in (34, 64, 66, 72, 128, 500)] + [(True, k) for k in (32, 34, 64, 128, 250, 500)])
@pytest.mark.parametrize("shape", [(4, 2, 132, 260), (6, 3, 260, 132), (4, 2, 40, 520), (6, 2, 2564, 2564), (40, 2, 130, 262), (4, 2, 128, 256)])
def test_fp16_parts(gpu, shape, k_first, k):
    batch, groups, n, m = shape
    if not k_first and (n % 4 or m % 4 or batch // groups > 16):
        n, m, batch = n // 4 * 4, m // 4 * 4, groups * 8
    if k_first and m == 132:
        m = 136                  # (rows of 8j + 4 elements: from 256 on)
    print("fp16 parts", batch, groups, n, m, k_first, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)
    A = torch.randn((batch, k, m) if k_first else (batch, m, k), generator=g, device="cuda").mul_(8).half()
    B = torch.randn((batch, k, n) if k_first else (batch, n, k), generator=g, device="cuda").mul_(8).half()
    parts = torch.full((groups, n, m), float("nan"), device="cuda")
    ck.gemm_fp16_parts(m, k, n, batch, groups, k_first, A.data_ptr(), B.data_ptr(), parts.data_ptr(), _st())
    p, q = (B.transpose(1, 2), A) if k_first else (B, A.transpose(1, 2))
    p, q, per = p.double().contiguous(), q.double().contiguous(), batch // groups
    for i in range(groups):
        want = sum(p[e] @ q[e] for e in range(i * per, (i + 1) * per))
        mag = sum(p[e].abs() @ q[e].abs() for e in range(i * per, (i + 1) * per))
        assert bool(((parts[i].double() - want).abs() <= mag * (per * k) * 2.0 ** -24).all()), (i, k)      # fp32 sums in any order
    if n * m % 4 == 0:
        _check_add(parts)


# (edges of the kernel for any size: rows of half pieces and of 4j + 2 elements, less than a tile, past one, several tiles of each width, operands off
# 16-byte boundaries; depths of a slab and less, a rest, many slabs; as many groups as entries)
@pytest.mark.parametrize("k", [2, 62, 64, 250])
@pytest.mark.parametrize("shape", [(6, 6, 8, 44), (4, 2, 6, 2), (9, 3, 66, 130), (20, 20, 126, 1030), (6, 2, 1002, 62), (300, 150, 4, 132), (6, 3, 260, 252)])
@pytest.mark.parametrize("at", [0, 1])
def test_fp16_parts_of_any_size(gpu, shape, k, at):
    batch, groups, n, m = shape
    print("fp16 parts of any size", shape, k, at, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)

    def operand(rows):
        flat = torch.randn(batch * k * rows + at, generator=g, device="cuda").mul_(8).half()
        return flat[at:].view(batch, k, rows)
    A, B = operand(m), operand(n)
    parts = torch.full((groups, n, m), float("nan"), device="cuda")
    ck.gemm_fp16_parts(m, k, n, batch, groups, 2, A.data_ptr(), B.data_ptr(), parts.data_ptr(), _st())
    p, q, per = B.double().transpose(1, 2).contiguous(), A.double(), batch // groups
    want, mag = (torch.stack([x[i] @ y[i] for i in range(batch)]).view(groups, per, n, m).sum(1) for x, y in ((p, q), (p.abs(), q.abs())))
    assert bool(((parts.double() - want).abs() <= mag * (per * k) * 2.0 ** -24).all())      # fp32 sums in any order
    _check_add(parts)


@pytest.mark.parametrize("batch,k,m,n", [(26, 128, 44, 8), (49, 128, 890, 136), (24, 980, 8, 28), (33, 836, 768, 128), (7, 66, 132, 260), (16, 64, 1024, 512), (5, 1024, 12, 48)])
def test_sum_of_krows_entries(gpu, batch, k, m, n):
    """Weight gradients of operands stored (K, rows): groups of any number of entries, none that leaves one workgroup a depth of thousands; sums in fp32, rounded once"""
    from cpm_kernels_amd.torch.gemm import gemm_pth_fp16_sum
    print("sum of (K, rows) entries", batch, k, m, n, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + m + k)
    A, B = (torch.randn((batch, k, r), generator=g, device="cuda").half() for r in (n, m))
    out = gemm_pth_fp16_sum(A, True, B, False).double()[0]
    p, q = A.double().transpose(1, 2).contiguous(), B.double()
    want, mag = (sum(x[i] @ y[i] for i in range(batch)) for x, y in ((p, q), (p.abs(), q.abs())))
    each = sum((p[i] @ q[i]).abs() for i in range(batch)) * 2.0 ** -11 if ck.gemm_sum_krows_groups(m, k, n, batch) == 0 else 0      # (one by one: each entry's rounding)
    assert bool(((out - want).abs() <= mag * (batch * k) * 2.0 ** -24 + each + want.abs() * 2.0 ** -10.9 + 2.0 ** -25).all())


def _check_add(parts):
    groups, total = parts.size(0), parts[0].numel()
    out = torch.full(parts.shape[1:], float("nan"), device="cuda", dtype=torch.half)
    ck.gemm_add_parts(groups, total, parts.data_ptr(), out.data_ptr(), _st())
    want, mag = parts.double().sum(0), parts.double().abs().sum(0)
    bound = mag * groups * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25
    big = want.abs() > 65504
    assert bool(((out.double() - want).abs() <= bound)[~big].all()) and bool((out[want.abs() > 65536].isinf()).all())


@pytest.mark.parametrize("groups,n", [(1, 4), (2, 4), (3, 1020), (7, 132), (64, 256), (200, 1028), (2, 1 << 21)])
def test_add_parts(gpu, groups, n):
    print("add parts", groups, n, flush=True)
    _check_add(torch.randn((groups, n), generator=torch.Generator(device="cuda").manual_seed(n + groups), device="cuda"))


@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("int8", [True, False])
def test_sums_that_pass_fp16_range_between_groups(gpu, int8, rows):
    """Entries that are finite each and cancel over the whole batch, while the sum of a group of them passes 65504."""
    import cpm_kernels_amd.torch as ct
    batch, tokens, size = 16, 128, 640
    groups = ck.gemm_sum_groups(size, size, batch)
    assert 1 < groups < batch
    print("range between groups", int8, rows, groups, flush=True)
    x = torch.full((batch, tokens, size) if rows else (batch, size, tokens), 16.0, device="cuda", dtype=torch.half)
    w = torch.full((1, size, size), 0.001, device="cuda", dtype=torch.half, requires_grad=True)
    out = ct.bmm(x, False, w, True, int8=int8) if rows else ct.bmm(w, False, x, False, int8=int8)
    grad = torch.full_like(out, 20.0)                 # 128 products of 16 x 20: 40960 an entry
    per = batch // groups
    for e in range(batch):
        if e // per % 2:
            grad[e] = -20.0
    got, = torch.autograd.grad(out, [w], grad)
    # equal entries of either sign cancel exactly, whatever their rounding, unless a partial sum was lost
    assert bool((got == 0).all()), got.flatten()[:4]
