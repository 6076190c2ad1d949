"""The block-scaled quantize and dequantize kernels of one mode and map each
(``vh_blockfast.h``, ``k_dequantize_blocks``) against the general kernels, bit
for bit and with the kernel that ran asserted: the same values behind a 16-byte
aligned address, which they need, and behind one that is not, over every form
they take, at edges of blocks, rows and workgroups, with zeros, NaN, infinities,
subnormal and huge blocks, quotients on rounding midpoints and scales that
saturate or flush their map; a case of each against the oracle."""

import pytest
import torch

import voyager_amd.library  # noqa: F401  (defines quantized_ops)
from helpers import assert_same_bits
from oracle import ops as O
from oracle import tables as T
from voyager_amd._lib import load

pytestmark = pytest.mark.gpu

# element map, block, largest value, scale map ("pot": powers of two; "affine")
FORMS = [("int8", 16, 127.0, "pot"), ("fp8_e4m3", 32, 448.0, "pot"), ("fp4_e2m1", 32, 6.0, "pot"),
         ("fp6_e3m2", 16, 28.0, "pot"), ("fp4_e2m1", 16, 6.0, "fp8_e4m3"), ("fp4_e2m1", 64, 6.0, "fp8_e5m3"),
         ("lut4_to_int6", 64, 31.0, "fp8_e5m3"), ("lut4_to_int6", 32, 31.0, "fp8_e4m3"),
         ("uint2", 32, 3.0, "affine_fp16_e5m10"), ("int4", 16, 7.0, "affine")]
# rows, columns: over 2**18 elements where the blocks run along a row, so that
# the one-element-a-lane kernels of small tensors do not take it; partial blocks
SHAPES = [(65, 4096), (300, 904), (77, 8200), (2, 131080)]


def _ran():
    return load().vh_last_kernel().decode()


def _unaligned(t):
    """The same values, two bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    view = flat[1:1 + t.numel()].view(t.shape)
    view.copy_(t)
    assert view.data_ptr() % 16 and view.is_contiguous()
    return view


def _values(rows, cols, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * torch.exp2(torch.randint(-20, 20, (rows, 1), generator=g).float())
    x = torch.where(torch.rand(rows, cols, generator=g) < 0.02, torch.round(x * 4) / 4, x)
    x[0, :128] = 0.0
    x[0, 128:256] = -0.0
    x[1, 5], x[1, 100], x[1, 200] = float("nan"), float("inf"), float("-inf")
    x[0, 256:320] = 1e-39
    x[0, 320:384] = 3e38
    x[0, 384:448] = torch.arange(64.0)
    x[0, 448:512] = 2.5
    x[-1, -8:] = -7.0
    return x.bfloat16().cuda()


def _tables(dtype, scale, dev="cuda"):
    t = T.quantization_map(dtype)
    mid = entries = None
    if dtype.startswith("lut"):
        t, entries, mid = T.codebook_index_table(t)
    name = scale.replace("affine_", "") if scale not in ("pot", "affine") else None
    s = None if name is None else T.quantization_map(name)
    return [None if v is None else v.to(dev) for v in (t, s, mid, entries)]


def _quantize(q, x, axis, form, tab, stab, mid):
    dtype, bs, qmax, scale = form
    if scale.startswith("affine"):
        return q.quantize_affine(x, tab, [axis], bs, 0.0 if dtype.startswith("u") else -8.0, qmax, stab)
    return q.quantize_mx(x, tab, [axis], bs, qmax, scale == "pot", stab, mid)


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"{f[0]}-{f[1]}-{f[3]}")
@pytest.mark.parametrize("axis", [-1, -2])
def test_same_as_general_kernels(form, axis):
    """... and back; only aligned tensors take the kernels under test."""
    q = torch.ops.quantized_ops
    tab, stab, mid, entries = _tables(form[0], form[3])
    for rows, cols in SHAPES:
        x = _values(rows, cols, rows)
        if axis == -2:
            x = x.mT.contiguous()
            if x.shape[-1] % 8:  # a multiple of eight inside the blocked dimension, which the column form needs
                x = torch.nn.functional.pad(x, (0, -x.shape[-1] % 8))
        fast = _quantize(q, x, axis, form, tab, stab, mid)
        assert _ran() == ("k_fast_rows" if axis == -1 else "k_fast_cols"), _ran()
        general = _quantize(q, _unaligned(x), axis, form, tab, stab, mid)
        # (MX integers along rows have a kernel of their own behind any address)
        own = axis == -1 and form[0].startswith("int") and form[3] == "pot"
        assert _ran() == ("k_mx_pot_int_rows8" if own else "k_rows" if axis == -1 else "k_cols"), _ran()
        for a, b, what in zip(fast, general, ("scale", "codes or zero point", "codes")):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), f"{what} of {list(x.shape)}"
        codes, scale = fast[-1], fast[0]

        def back(c):
            if form[3].startswith("affine"):
                return q.dequantize(c, scale, fast[1], [axis], form[1])
            return q.dequantize_mx(c, scale, form[1], entries)

        one, ran = back(codes), _ran()
        two = back(_unaligned(codes))
        assert (ran, _ran()) == ("k_dequantize_blocks", "k_dequantize"), list(x.shape)
        assert torch.equal(one.view(torch.int16), two.view(torch.int16)), f"dequantize of {list(x.shape)}"


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"{f[0]}-{f[1]}-{f[3]}")
@pytest.mark.parametrize("axis", [-1, -2])
def test_same_as_oracle(form, axis):
    q = torch.ops.quantized_ops
    x = _values(72, 4104, 3)
    tab, stab, mid, _ = _tables(form[0], form[3])
    got = _quantize(q, x, axis, form, tab, stab, mid)
    assert _ran() == ("k_fast_rows" if axis == -1 else "k_fast_cols"), _ran()
    ctab, cstab, cmid, _ = _tables(form[0], form[3], "cpu")
    exp = _quantize(O, x.cpu(), axis, form, ctab, cstab, cmid)
    for a, b, what in zip(got, exp, ("scale", "codes or zero point", "codes")):
        assert_same_bits(a, b, what)


@pytest.mark.parametrize("shape,axis", [((3, 5, 96, 128), -2), ((3, 5, 96, 128), -1), ((3, 5, 50, 24), -2),
                                        ((2, 100, 8, 16), 1), ((4, 33), -1)])
def test_dequantize_layouts(shape, axis):
    """Blocks along any dimension with and without zero points, odd codes
    (NaN, infinities), and a scalar scale, aligned against unaligned."""
    q = torch.ops.quantized_ops
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(*shape, generator=g)
    x.view(-1)[::97] = float("nan")
    x.view(-1)[::101] = float("inf")
    x = x.bfloat16().cuda()
    ps = list(shape)
    ps[axis] = -(-ps[axis] // 32)
    s, z = (torch.randn(*ps, generator=g).bfloat16().cuda() for _ in range(2))
    one = torch.tensor(0.37, device="cuda")
    for args in ((s, z, [axis], 32), (s, None, [axis], 32), (one,), (one.bfloat16(),)):
        a, ran = q.dequantize(x, *args), _ran()
        b = q.dequantize(_unaligned(x), *args)
        assert _ran() == "k_dequantize"
        assert ran == ("k_dequantize_blocks" if shape[-1] % 8 == 0 else "k_dequantize"), args[2:]
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), args[2:]


@pytest.mark.parametrize("rows", [1, 2, 3])
def test_few_affine_rows(rows):
    """A token or two into a cache's column blocks, on the general kernel."""
    q = torch.ops.quantized_ops
    form = FORMS[8]
    tab, stab, mid, _ = _tables(form[0], form[3])
    x = torch.randn(3, rows, 128, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
    got = _quantize(q, x, -2, form, tab, stab, mid)
    assert _ran() == ("k_cols" if rows <= 2 else "k_fast_cols")
    ctab, cstab, _, _ = _tables(form[0], form[3], "cpu")
    for a, b, what in zip(got, _quantize(O, x.cpu(), -2, form, ctab, cstab, None), ("scale", "zero point", "codes")):
        assert_same_bits(a, b, what)
