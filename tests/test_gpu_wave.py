"""GPU: the wave kernels (k_gemv_wave, k_decode_wave), which serve 1024-weight
blocks of every profile where the sip and gulp kernels do not: columns that
are not whole blocks, the balanced profile, fp32 activations. Against the
oracle, at the sizes where their split can go wrong: one weight, one row, odd
row counts (a unit's second row missing), a last block of 1, 4 and 1023
weights, columns that are not dword-aligned, one block a row, more units than
one directory read (32) a wave; and at escape densities from none to past
every limit of the in-register tiers (512 tier-0 and 128 tier-1 escapes, 64
tail words), which take the reads from memory; and at each such limit, one past
it, and with every weight escaping as far as each tier."""

import zlib

import numpy as np
import pytest

from oracle import radix_oracle as O
from tests.helpers import bf16_tensor, escape_heavy_bits, finite_bits, pack_to_dict, u16_of

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1025), (3, 1028), (5, 2047), (130, 260), (17, 3079), (1000, 2052), (1030, 9476), (97, 20484)]


def _bits(rng, kind, shape):
    if kind == "tight":
        return finite_bits(rng, shape)
    if kind == "spread":
        return finite_bits(rng, shape, spread=True)
    return escape_heavy_bits(rng, shape, {"none": 0.0, "dense": 0.35}[kind])


@pytest.mark.parametrize("profile", ["sip", "balanced", "gulp"])
@pytest.mark.parametrize("shape", SHAPES)
def test_decode_and_gemv_against_the_oracle(cuda, profile, shape):
    import torch

    from drinkme_amd import radix_ops, swap

    R, C = shape
    rng = np.random.default_rng(zlib.crc32(repr((profile, shape)).encode()))
    for kind in ("tight", "spread", "none", "dense"):
        bits = _bits(rng, kind, shape)
        p = O.pack(bits, profile, allow_raw=False)
        rt = swap.to_device_radix(pack_to_dict(p, profile), cuda)
        print(f"case wave {profile} {shape} {kind}", flush=True)
        assert np.array_equal(u16_of(radix_ops.decode_bits(rt)), bits), kind
        xf = rng.standard_normal((8, C)).astype(np.float32)
        for dtype in (torch.float32, torch.bfloat16):
            # (rows starting one element into a buffer: the bf16 ones are not dword-aligned)
            buf = torch.empty(8 * C + 1, dtype=dtype, device=cuda)
            x = buf[1:].view(8, C)
            x.copy_(torch.from_numpy(xf))
            ref, bound = O.gemv_f64(bits, x.float().cpu().numpy())
            rows = radix_ops.gemv_rows(rt, x, None, torch.float32)
            err = np.abs(rows.cpu().numpy().astype(np.float64) - ref) / bound
            assert err.max() <= 1.0, f"{kind} {dtype}: err/bound {err.max():.3g}"
            # every row the same at any M and alignment, up to the kernels' own order of sums where
            # bf16 rows of whole blocks run elsewhere (no shape here has whole blocks)
            for M in (1, 2, 3, 5):
                assert torch.equal(radix_ops.gemv_rows(rt, x[:M].clone(), None, torch.float32), rows[:M]), f"{kind} M={M}"
            bias = torch.from_numpy(rng.standard_normal(R).astype(np.float32)).to(cuda)
            fused = radix_ops.gemv_rows(rt, x[:2], bias, torch.bfloat16)
            assert torch.equal(fused, (rows[:2] + bias).to(torch.bfloat16)), f"{kind}: fused epilogue"


@pytest.mark.parametrize("profile,dtype", [("sip", "float32"), ("balanced", "bfloat16"), ("gulp", "float32")])
def test_whole_blocks_and_groups(cuda, profile, dtype):
    """Whole-block columns (their fp32 and balanced route) and a group of
    three tensors in one launch: each output is its own launch's, bit for
    bit."""
    import torch

    from drinkme_amd import radix_ops, swap

    rng = np.random.default_rng(zlib.crc32((profile + dtype).encode()))
    C = 4096
    ps, srcs = [], []
    for R in (1027, 64, 2):
        bits = finite_bits(rng, (R, C), spread=True)
        srcs.append(bits)
        ps.append(swap.to_device_radix(pack_to_dict(O.pack(bits, profile, allow_raw=False), profile), cuda))
    for M in (1, 4, 7):
        x = torch.from_numpy(rng.standard_normal((M, C)).astype(np.float32)).to(cuda).to(getattr(torch, dtype))
        print(f"case wave group {profile} {dtype} M={M}", flush=True)
        outs = radix_ops.gemv_group(ps, x, None, torch.float32)
        for p, bits, y in zip(ps, srcs, outs):
            assert torch.equal(y, radix_ops.gemv_rows(p, x, None, torch.float32))
            ref, bound = O.gemv_f64(bits, x.float().cpu().numpy())
            assert np.all(np.abs(y.cpu().numpy().astype(np.float64) - ref) <= bound)


def test_a_non_finite_weight_past_the_row_end_is_not_multiplied(cuda):
    """Palette entry 0 is the exponent of infinities here: the lanes past a
    row's last column must not bring it (0 x inf) into the sums."""
    import torch

    from drinkme_amd import radix_ops, swap

    rng = np.random.default_rng(5)
    bits = finite_bits(rng, (8, 1028))
    bits[:6, :1024] = 255 << 7  # six rows of infinities, two finite ones
    x = torch.ones(1, 1028, device=cuda)
    for profile in ("sip", "balanced", "gulp"):
        rt = swap.to_device_radix(pack_to_dict(O.pack(bits, profile, allow_raw=False), profile), cuda)
        assert rt["rx_palette_np"][0] == 255
        assert np.array_equal(u16_of(radix_ops.decode_bits(rt)), bits)
        for xx in (x, x.to(torch.bfloat16)):
            y = radix_ops.gemv_rows(rt, xx, None, torch.float32).cpu().numpy()[0]
            assert np.all(np.isinf(y[:6])) and np.all(np.isfinite(y[6:])), profile


@pytest.mark.parametrize("M,blocks", [(1, 2047), (1, 2049), (2, 1025), (3, 512), (4, 513), (2, 4), (4, 1)])
def test_gulp_rows_at_the_edge_of_the_wave_kernels_sums(cuda, M, blocks):
    """Whole-block gulp at up to four rows runs the wave kernel while two
    rows' sums fit it (2048 / M column blocks, M rounded up to a power of
    two), the gulp kernel beyond; three rows of weights, the second of the
    last unit missing. The twin follows bit for bit on either side of the
    edge, and on the wave kernel's from a weight that is not 16-byte aligned
    too (the gulp kernel's twin needs that alignment)."""
    import torch

    from drinkme_amd import radix_ops, swap

    R, C = 3, 1024 * blocks
    rng = np.random.default_rng(blocks + M)
    bits = escape_heavy_bits(rng, (R, C), 0.05)
    rt = swap.to_device_radix(pack_to_dict(O.pack(bits, "gulp", allow_raw=False), "gulp"), cuda)
    xb = O.f32_to_bf16_bits(rng.standard_normal((M, C)).astype(np.float32))
    x = bf16_tensor(xb, cuda)
    print(f"case wave gulp edge M={M} blocks={blocks}", flush=True)
    y = radix_ops.gemv_rows(rt, x, None, torch.float32)
    ref, bound = O.gemv_f64(bits, O.bf16_bits_to_f32(xb))
    assert np.all(np.abs(y.cpu().numpy().astype(np.float64) - ref) <= bound)
    buf = torch.empty(R * C + 2, dtype=torch.bfloat16, device=cuda)
    for start in (0, 2) if blocks * (M if M < 3 else 4) <= 2048 else (0,):
        w = buf[start:start + R * C].view(R, C)
        w.copy_(bf16_tensor(bits, cuda))
        twin = dict(swap.to_device_twin(w, widths=rt["widths"], device=cuda), weight=w)
        assert torch.equal(radix_ops.gemv_rows(twin, x, None, torch.float32), y), start


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("profile", ["sip", "balanced", "gulp"])
def test_the_generic_kernel_on_the_wave_kernels_tensors(cuda, profile, dtype):
    """Other block sizes and rows past the wave kernel's sums still run it."""
    import torch

    from drinkme_amd import radix_ops, swap

    for R, C in ((130, 260), (17, 3079), (64, 2048)):
        rng = np.random.default_rng(R + C)
        bits = finite_bits(rng, (R, C), spread=True)
        rt = swap.to_device_radix(pack_to_dict(O.pack(bits, profile, allow_raw=False), profile), cuda)
        x = torch.from_numpy(rng.standard_normal((8, C)).astype(np.float32)).to(cuda).to(getattr(torch, dtype))
        ref, bound = O.gemv_f64(bits, x.float().cpu().numpy())
        print(f"case wave generic {profile} {dtype} {(R, C)}", flush=True)
        prev = radix_ops.set_policy("generic")
        try:
            for M in range(1, 9):
                y = radix_ops.gemv_rows(rt, x[:M], None, torch.float32).cpu().numpy().astype(np.float64)
                assert np.all(np.abs(y - ref[:M]) <= bound[:M]), f"{(R, C)} M={M}"
        finally:
            radix_ops.set_policy(prev)


# (escapes of tier 0, of tier 1, of tier 2) of a block, by profile: none, the in-register tiers' limits (sip 256
# terminal bytes; 512 and 128 escapes; 64 tail words) and one past each, every weight escaping as far as each tier
COUNTS = {
    "sip": [(0,), (1,), (255,), (256,), (257,), (700,), (1024,)],
    "balanced": [(0, 0), (512, 60), (512, 64), (512, 65), (513, 0), (170, 180 - 12), (600, 600), (1024, 0),
                 (1024, 1024), (1024, 1)],
    "gulp": [(0, 0, 0), (512, 128, 64), (512, 128, 65), (512, 129, 0), (513, 0, 0), (512, 0, 0), (128, 128, 128),
             (700, 300, 40), (1024, 0, 0), (1024, 1024, 0), (1024, 1024, 1024), (1024, 1, 1), (129, 129, 129)],
}
TIERS = {"sip": (7,), "balanced": (3, 7), "gulp": (3, 3, 15)}


def _counted_bits(rng, profile, cols):
    """Rows whose every 1024-weight block has the escape counts of one entry
    of COUNTS (each next to each: a unit with one such row, and with two),
    then rows that fix the palette's order."""
    sizes = (*TIERS[profile], 19)
    start = np.cumsum((0, *sizes))
    exps = [125 - np.arange(start[t], start[t + 1]) for t in range(len(sizes))]

    def block(counts):
        left = 1024
        tier = np.empty(1024, np.int64)
        for t, c in enumerate((*counts, 0)):
            c = min(c, left)
            tier[c:left], left = t, c
        rng.shuffle(tier)
        return np.concatenate([exps[t][rng.integers(0, sizes[t], 1024)][:, None] for t in range(len(sizes))],
                              axis=1)[np.arange(1024), tier]

    nb = -(-cols // 1024)
    rows = [np.concatenate([block(c) for _ in range(nb)])[:cols] for c in COUNTS[profile] for _ in range(2)]
    rows += [rows[i] for i in rng.permutation(len(rows))]
    share = {1: (.94, .06), 2: (.75, .22, .03), 3: (.65, .26, .08, .01)}[len(sizes) - 1]
    every = np.concatenate(exps)
    p = np.concatenate([np.full(n, s / n) for n, s in zip(sizes, share)])
    filler = rng.choice(every, size=(len(rows) * 12, cols), p=p)
    e = np.concatenate([np.array(rows), filler]).astype(np.uint16)
    return (e << 7) | rng.integers(0, 128, e.shape, dtype=np.uint16) | (rng.integers(0, 2, e.shape, dtype=np.uint16) << 15), exps


@pytest.mark.parametrize("cols", [2048, 1024 + 1000])
@pytest.mark.parametrize("profile", ["sip", "balanced", "gulp"])
def test_blocks_at_and_past_the_limits_of_the_in_register_tiers(cuda, profile, cols):
    import torch

    from drinkme_amd import radix_ops, swap

    rng = np.random.default_rng(zlib.crc32(repr((profile, cols)).encode()))
    bits, exps = _counted_bits(rng, profile, cols)
    p = O.pack(bits, profile, allow_raw=False)
    at = 0
    for tier in exps[:-1]:  # the tiers' exponents are those the counts were made for
        assert set(p.palette.reshape(-1)[at:at + len(tier)]) == set(tier)
        at += len(tier)
    rt = swap.to_device_radix(pack_to_dict(p, profile), cuda)
    print(f"case wave counts {profile} {cols}", flush=True)
    assert np.array_equal(u16_of(radix_ops.decode_bits(rt)), bits)
    xf = rng.standard_normal((8, cols)).astype(np.float32)
    for dtype, M in ((torch.bfloat16, 1), (torch.bfloat16, 4), (torch.float32, 2), (torch.float32, 8)):
        x = torch.from_numpy(xf[:M]).to(cuda).to(dtype)
        ref, bound = O.gemv_f64(bits, x.float().cpu().numpy())
        y = radix_ops.gemv_rows(rt, x, None, torch.float32).cpu().numpy().astype(np.float64)
        assert np.all(np.abs(y - ref) <= bound), f"{dtype} M={M}"


def test_rows_of_different_scale_stay_near_the_unscaled_time(cuda):
    """One palette over rows whose scales differ by a lognormal of sigma 0.5
    puts a fifth of gulp's units past the in-register limits. Measured 1.5
    times the unscaled launch; 4.3 on the gulp kernel, 7.8 where such blocks
    are read a field at a time. The bound, 3, stands between."""
    import torch

    from drinkme_amd import radix_ops, radix_pack, swap

    R, C = 12288, 4096
    gen = torch.Generator(device=cuda).manual_seed(7)
    w = torch.randn(R, C, generator=gen, device=cuda) * 0.02
    scale = torch.exp(0.5 * torch.randn(R, 1, generator=gen, device=cuda))
    x = torch.randn(1, C, generator=gen, device=cuda).to(torch.bfloat16)
    took = []
    for weight in (w, w * scale):
        bits = u16_of(weight.to(torch.bfloat16))
        call = radix_ops.RowsLauncher(swap.to_device_radix(radix_pack.pack_array_radix(bits, "gulp"), cuda))
        best = float("inf")
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            call(x)
            a.record()
            for _ in range(50):
                call(x)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        took.append(best)
    assert took[1] < 3 * took[0], took
