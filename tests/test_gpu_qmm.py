"""GPU: PrefillInt4QMM (dense int4 projection over t tokens) through the C-ABI,
against the oracle (fp16-staged weights, exact sums) within the north-star
1e-3 relative bound, at the Gemma projection shapes and ragged token counts.
Output rows past t stay untouched. Declines and errors as documented."""
import numpy as np
import pytest

import oracle
from tests import kernelcheck as kc
from tests.gpu_util import dev, empty, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tsg():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import tsugumi_amd
    return tsugumi_amd


def operands(rng, n, k, g):
    packed = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    scales = oracle.bf16_bits((np.abs(rng.normal(0, 0.02, n * (k // g))) / 7).astype(np.float32))
    biases = oracle.bf16_bits(rng.normal(0, 0.01, n * (k // g)).astype(np.float32))
    return packed, scales, biases


@pytest.mark.parametrize("t,n,k,g,scheme", [
    (1, 2816, 2816, 64, "affine"), (37, 4096, 2816, 32, "sym"), (300, 2816, 4096, 64, "sym"),
    (2048, 2816, 2816, 32, "affine"), (129, 704, 2816, 32, "sym"), (255, 8192, 2816, 64, "affine"),
    (2048, 4096, 2816, 32, "sym"),
])
def test_qmm_matches_oracle(tsg, t, n, k, g, scheme):
    print(f"qmm t={t} n={n} k={k} g{g} {scheme}", flush=True)
    sym = scheme == "sym"
    ctx = tsg.Context(0, group_size=g)
    ctx.set_affine_scheme(scheme)
    rng = np.random.default_rng(t * 7 + n)
    packed, scales, biases = operands(rng, n, k, g)
    xb = oracle.f16_bits(rng.normal(0, 1, t * k).astype(np.float32))
    y = empty(t * n + 64, fill=0x1234)
    tsg.PrefillInt4QMM(ctx).encode(dev(packed), dev(scales), None if sym else dev(biases),
                                   dev(xb), y, t, n, k)
    got = host(y, np.uint16)
    assert np.all(got[t * n:] == 0x1234)
    ref = oracle.int4_qmm(packed, scales, None if sym else biases, xb, t, n, k, g, sym)
    rel = oracle.relative_error(oracle.f16_to_float(got[:t * n]),
                                oracle.f16_to_float(ref.ravel()))
    print(f"  rel={rel:.3e}")
    assert rel <= kc.NORTH_STAR
    ctx.close()


@pytest.mark.parametrize("scheme", ["sym", "affine"])
def test_qmm_narrow_tiles_equal_wide_tiles_bitwise(tsg, scheme):
    """Below 256 workgroups of 256 columns the QMM runs 128-column tiles (one
    weight tile per wave); each column keeps the same MFMA sequence, so the
    results are the wide tiles' bit for bit. T = 2048: N = 4096 runs 256 wide
    workgroups, its first 2816 weight rows as N = 2816 176 -> 352 narrow ones;
    the shared 2816 columns must agree exactly."""
    t, k, g, n_wide, n_narrow = 2048, 2816, 32, 4096, 2816
    print(f"qmm narrow vs wide {scheme}", flush=True)
    sym = scheme == "sym"
    ctx = tsg.Context(0, group_size=g)
    ctx.set_affine_scheme(scheme)
    rng = np.random.default_rng(4242 + sym)
    packed, scales, biases = operands(rng, n_wide, k, g)
    xb = oracle.f16_bits(rng.normal(0, 1, t * k).astype(np.float32))
    q = tsg.PrefillInt4QMM(ctx)
    y_wide, y_narrow = empty(t * n_wide), empty(t * n_narrow)
    sg = n_narrow * (k // g)
    q.encode(dev(packed), dev(scales), None if sym else dev(biases), dev(xb), y_wide, t, n_wide, k)
    q.encode(dev(np.ascontiguousarray(packed[:n_narrow])), dev(scales[:sg].copy()),
             None if sym else dev(biases[:sg].copy()), dev(xb), y_narrow, t, n_narrow, k)
    wide = host(y_wide, np.uint16).reshape(t, n_wide)[:, :n_narrow]
    narrow = host(y_narrow, np.uint16).reshape(t, n_narrow)
    assert np.array_equal(wide, narrow)
    ctx.close()


def test_qmm_errors(tsg):
    ctx = tsg.Context(0, group_size=32)
    q = tsg.PrefillInt4QMM(ctx)
    w, s, x, y = empty(64 * 64), empty(64 * 8), empty(4 * 256), empty(4 * 64)
    with pytest.raises(tsg.TsgError) as e:
        q.encode(w, s, s, x, y, 4, 64, 100)          # K % group
    assert e.value.status == 1 and "multiple of 32" in str(e.value)
    with pytest.raises(tsg.TsgError) as e:
        q.encode(w, s, s, x, y, 4, 48, 256)          # N % 64: the tiled path declines
    assert e.value.status == 3
    with pytest.raises(tsg.TsgError) as e:
        q.encode(w, s, s, x[1:], y, 4, 64, 256)      # x misaligned
    assert e.value.status == 2
    with pytest.raises(tsg.TsgError) as e:
        q.encode(w, s, s, x, y, 0, 64, 256)
    assert e.value.status == 1
    ctx.close()


@pytest.mark.parametrize("g,scheme", [(32, "sym"), (64, "affine")])
@pytest.mark.parametrize("t,n,k", [(300, 8192, 2048), (300, 8192, 704)])
def test_qmm_tables_at_the_end_of_an_allocation(tsg, t, n, k, g, scheme):
    """The scale and bias tables end where their allocations end (whole 2 MiB
    pages of their own): the last weight row's windows, which reach past its
    groups, read nothing behind the table."""
    import torch
    print(f"qmm tables at the end t={t} n={n} k={k} g{g} {scheme}", flush=True)
    sym = scheme == "sym"
    ctx = tsg.Context(0, group_size=g)
    ctx.set_affine_scheme(scheme)
    rng = np.random.default_rng(k + g)
    packed, scales, biases = operands(rng, n, k, g)
    xb = oracle.f16_bits(rng.normal(0, 1, t * k).astype(np.float32))

    def at_end(bits):
        page = torch.zeros(12 << 20, dtype=torch.uint8, device="cuda")
        tail = page[page.numel() - bits.nbytes:]
        tail.copy_(torch.from_numpy(np.ascontiguousarray(bits).view(np.uint8).copy()))
        return tail

    y = empty(t * n)
    tsg.PrefillInt4QMM(ctx).encode(dev(packed), at_end(scales), None if sym else at_end(biases),
                                   dev(xb), y, t, n, k)
    ref = oracle.int4_qmm(packed, scales, None if sym else biases, xb, t, n, k, g, sym)
    assert oracle.relative_error(oracle.f16_to_float(host(y, np.uint16)),
                                 oracle.f16_to_float(ref.ravel())) <= kc.NORTH_STAR
    ctx.close()


@pytest.mark.parametrize("g,scheme", [(32, "sym"), (32, "affine"), (64, "sym"), (64, "affine")])
@pytest.mark.parametrize("t,n,k", [(1, 64, 64), (31, 64, 448), (32, 128, 512), (33, 192, 576),
                                   (65, 64, 2112), (67, 4096, 2816)])
def test_qmm_of_few_rows(tsg, t, n, k, g, scheme):
    """The K-split kernel at the edges of its row blocks (1 to 67 rows) and of
    its deal of chunks (fewer than the waves, one round, one more, the read-ahead
    and past it), against fp64 over the kernel's fp16 weights: one fp16 rounding
    of each result (2^-11 of it) and K fp32 roundings (K 2^-24 of the sum of
    the magnitudes). The rows past y keep their bytes."""
    print(f"qmm few rows t={t} n={n} k={k} g{g} {scheme}", flush=True)
    check_elements(tsg, t, n, k, g, scheme)


def check_elements(tsg, t, n, k, g, scheme, in_place=False):
    """Every element against fp64, in the bound of test_qmm_of_few_rows; y past
    t rows keeps its bytes. in_place: y is x's buffer (n == k)."""
    sym = scheme == "sym"
    ctx = tsg.Context(0, group_size=g)
    ctx.set_affine_scheme(scheme)
    rng = np.random.default_rng(t + n + k)
    packed, scales, biases = operands(rng, n, k, g)
    xb = oracle.f16_bits(rng.normal(0, 1, t * k).astype(np.float32))
    y = empty(t * n + 64, fill=0x1234)
    x_dev = y if in_place else dev(xb)
    if in_place:
        y[:t * k] = dev(xb)
    tsg.PrefillInt4QMM(ctx).encode(dev(packed), dev(scales), None if sym else dev(biases),
                                   x_dev, y, t, n, k)
    got = host(y, np.uint16)
    assert np.all(got[t * n:] == 0x1234)
    s = np.repeat(oracle.bf16_to_float(scales).reshape(n, k // g).astype(np.float32), g, axis=1)
    b = (np.float32(-8) * s if sym else
         np.repeat(oracle.bf16_to_float(biases).reshape(n, k // g).astype(np.float32), g, axis=1))
    q = np.stack([packed & 15, packed >> 4], axis=-1).reshape(n, k)
    # q s is exact in fp64, q s + b rounds there before fp32: twice, at most 1 ulp
    w = (q.astype(np.float64) * s + b).astype(np.float32).astype(np.float16).astype(np.float64)
    x = oracle.f16_to_float(xb).reshape(t, k).astype(np.float64)
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    err = np.abs(oracle.f16_to_float(got[:t * n]).reshape(t, n) - ref)
    assert np.all(err <= np.abs(ref) * 2.0 ** -11 + mag * k * 2.0 ** -24 + 2.0 ** -25)
    ctx.close()


@pytest.mark.parametrize("g,scheme", [(32, "sym"), (64, "affine")])
@pytest.mark.parametrize("t,n,k", [(1025, 2880, 704), (1100, 2880, 2816), (1100, 2880, 704),
                                   (2049, 4160, 704), (2112, 4160, 704)])
def test_qmm_gemm_at_ragged_tiles(tsg, t, n, k, g, scheme):
    """The GEMM at row blocks of 1, 64 and 76 rows past full ones (one, two and
    three slices) and at a last column tile of 64 live columns: 128-column tiles
    (n = 2880) and 256-column ones, three of whose waves are dead (n = 4160 from
    2049 rows), per element."""
    print(f"qmm gemm ragged t={t} n={n} k={k} g{g} {scheme}", flush=True)
    check_elements(tsg, t, n, k, g, scheme)


@pytest.mark.parametrize("t,n", [(100, 128), (200, 64)])
def test_qmm_in_place(tsg, t, n):
    """y in x's buffer where one column tile holds all columns: each row block
    has read its rows when it writes them. Few rows as these go to the K split
    otherwise, whose workgroups would read rows that others have written."""
    print(f"qmm in place t={t} n={n}", flush=True)
    check_elements(tsg, t, n, n, 32, "sym", in_place=True)


@pytest.mark.parametrize("t,n,k,g,scheme", [
    (32, 704, 512, 32, "sym"), (130, 704, 512, 32, "affine"), (32, 2048, 384, 64, "affine"),
    (25, 704, 256, 32, "sym"), (40, 2048, 448, 64, "affine"), (32, 8256, 2560, 32, "affine"),
    (25, 16384, 2112, 32, "sym"), (64, 4160, 3584, 32, "sym"), (36, 8192, 2560, 32, "affine"),
    (96, 5440, 3584, 32, "affine"), (64, 8192, 4096, 64, "affine"),
])
def test_qmm_rows_past_the_split_keep_the_gemms_bits(tsg, t, n, k, g, scheme):
    """Few rows that the K split once took although the GEMM is the faster:
    their rows are those of a call of 2048 rows, bit for bit (the GEMM's sum does
    not depend on the rows beside a row)."""
    print(f"qmm past the split t={t} n={n} k={k} g{g} {scheme}", flush=True)
    import torch
    sym = scheme == "sym"
    ctx = tsg.Context(0, group_size=g)
    ctx.set_affine_scheme(scheme)
    rng = np.random.default_rng(t + n + k)
    packed, scales, biases = operands(rng, n, k, g)
    x = dev(oracle.f16_bits(rng.normal(0, 1, 2048 * k).astype(np.float32)))
    W, S, B = dev(packed), dev(scales), None if sym else dev(biases)
    few, many = empty(t * n), empty(2048 * n)
    q = tsg.PrefillInt4QMM(ctx)
    q.encode(W, S, B, x, few, t, n, k)
    q.encode(W, S, B, x, many, 2048, n, k)
    assert torch.equal(few, many[:t * n])
    ctx.close()
