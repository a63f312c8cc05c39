"""GPU parity of exl3r_gumbel_noise and exl3r_gumbel_sample against the CPU oracle (itself pinned by
the Philox known-answer vectors, an exhaustive accuracy check of the noise transform and the
Gumbel-max distribution): bit-exact noise and exactly equal token ids on decode and prefill logits,
every dtype, the max_logit mask, unaligned rows, special values, zero rows, and the identity
gumbel_sample(x) == argmax_sample(gumbel_noise(x)) on the device."""
import math

import numpy as np
import pytest
import torch

import exl3r.ffi as ffi
from _gpu import NTHREADS, TORCH_DT, dev_normal, from_dev, graph_us, to_dev
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

F16, BF16, F32 = orc.F16, orc.BF16, orc.F32


def run_sample(logits, dt, seed, max_logit=0):
    ids = torch.full((logits.shape[0],), -7, dtype=torch.int64, device="cuda")
    ffi.gumbel_sample(logits, ids, max_logit, seed)
    torch.cuda.synchronize()
    exp = orc.gumbel_sample(np.ascontiguousarray(from_dev(logits)), dt, seed, max_logit, nthreads=NTHREADS)
    got = ids.cpu().numpy()
    assert np.array_equal(got, exp), f"rows differing: {np.nonzero(got != exp)[0][:8]}"
    return got


def run_noise(x, dt, seed, out_dt):
    out = torch.empty(x.shape, dtype=TORCH_DT[out_dt], device="cuda")
    ffi.gumbel_noise(x, out, seed)
    torch.cuda.synchronize()
    exp = orc.gumbel_noise(np.ascontiguousarray(from_dev(x)), dt, seed, out_dt, nthreads=NTHREADS)
    got = from_dev(out)
    same = (got.view(np.uint32) == exp.view(np.uint32)) if out_dt == F32 else (got == exp)
    assert same.all(), f"{(~same).sum()} elements differ, first at {np.argwhere(~same)[:4].tolist()}"


@pytest.mark.parametrize("rows", [1, 8, 64])
def test_sample_decode_vocab(rows):
    run_sample(dev_normal((rows, 151936), 0, 3, F16, 40 + rows), F16, 1234 + rows)


@pytest.mark.parametrize("dt", [BF16, F32])
def test_sample_prefill_rows(dt):
    run_sample(dev_normal((600, 32000), 0, 3, dt, 41), dt, 77)          # row-per-workgroup kernel


@pytest.mark.parametrize("rows", [383, 384])
def test_sample_kernel_switch(rows):
    run_sample(dev_normal((rows, 9001), 0, 3, F16, 49), F16, 78)


@pytest.mark.parametrize("m", [1, 2, 151643, 151936, 200000])
def test_sample_mask(m):
    ids = run_sample(dev_normal((4, 151936), 0, 1, F16, 42), F16, 5, m)
    assert ids.max() < min(m, 151936)


def test_sample_special_values_and_unaligned():
    x = np.full((6, 3001), -1.0, np.float32)
    x[0, :] = -np.inf
    x[1, 2500] = np.inf
    x[2, [7, 2999]] = np.nan
    x[3, 1500] = 40.0               # 40 - 2.82 beats -1 + 16.64: always drawn
    x[5, :] = 0.0
    for dt in (F16, F32):
        got = run_sample(to_dev(orc.to_bits(x, dt), dt), dt, 9)
        assert list(got[:4]) == [got[0], 2500, 7, 1500]
    base = dev_normal((5, 4097), 0, 3, BF16, 43)
    run_sample(base[:, 1:], BF16, 10)                  # 2 bytes off 16-byte alignment: element path
    run_sample(base[:, :4001], BF16, 11, 3999)         # odd stride 4097


@pytest.mark.parametrize("seed", [0, 0xFFFFFFFF])
def test_sample_seeds(seed):
    run_sample(dev_normal((16, 50000), 0, 2, F16, 44), F16, seed)


@pytest.mark.parametrize("xt,ot", [(F16, F32), (BF16, F32), (F32, F32), (F16, F16), (F32, BF16)])
def test_noise_dtypes(xt, ot):
    run_noise(dev_normal((9, 8200), 0, 3, xt, 45), xt, 31337, ot)


def test_noise_unaligned_odd_and_in_place():
    base = dev_normal((7, 1001), 0, 3, F32, 46)
    run_noise(base[:, 1:], F32, 3, F32)
    run_noise(base[:, :999], F32, 4, F16)
    x = dev_normal((3, 4096), 0, 3, F32, 47)
    exp = orc.gumbel_noise(from_dev(x), F32, 8, F32)
    ffi.gumbel_noise(x, x, 8)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(x).view(np.uint32), exp.view(np.uint32))


def test_sample_equals_argmax_of_noise_on_device():
    x = dev_normal((64, 151936), 0, 3, F16, 48)
    noisy = torch.empty(x.shape, dtype=torch.float32, device="cuda")
    ffi.gumbel_noise(x, noisy, 2024)
    a = torch.empty(64, dtype=torch.int64, device="cuda")
    b = torch.empty(64, dtype=torch.int64, device="cuda")
    ffi.argmax_sample(noisy, a, 100000)
    ffi.gumbel_sample(x, b, 100000, 2024)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_draws_follow_softmax():
    logits = torch.tensor([0.0, 1.0, 2.0, -1.0, 0.5, 3.0, float("-inf"), 2.0, -4.0], device="cuda")
    rows = 200000
    ids = torch.empty(rows, dtype=torch.int64, device="cuda")
    ffi.gumbel_sample(logits.expand(rows, -1).contiguous(), ids, 0, 99)
    counts = torch.bincount(ids, minlength=9).double().cpu().numpy()
    p = torch.softmax(logits.double(), 0).cpu().numpy()
    live = p > 0
    assert counts[~live].sum() == 0
    e = p[live] * rows
    chi2 = float(((counts[live] - e) ** 2 / e).sum())
    dof = int(live.sum()) - 1
    assert chi2 < dof + 6 * math.sqrt(2 * dof), chi2


def test_zero_rows_and_cols():
    ids = torch.empty(0, dtype=torch.int64, device="cuda")
    ffi.gumbel_sample(torch.empty((0, 100), device="cuda", dtype=torch.float16), ids, 0, 1)
    x = torch.empty((0, 64), device="cuda")
    ffi.gumbel_noise(x, x, 1)
    y = torch.empty((4, 0), device="cuda")
    ffi.gumbel_noise(y, y, 1)
    torch.cuda.synchronize()


@pytest.mark.parametrize("rows,vocab,width", [(1, 151936, 0.0), (16, 40961, 1e-5), (64, 151936, 1e-4), (400, 20011, 3e-6)])
def test_sample_near_ties(rows, vocab, width):
    """Logits that undo the noise to within `width` (0: to the rounding of the sum), so that almost every
    candidate comes within the bound that decides which ones the draw evaluates exactly, on both kernels and on
    rows of every alignment.  The draw is the oracle's, which evaluates all of them."""
    noise = torch.empty((rows, vocab), dtype=torch.float32, device="cuda")
    ffi.gumbel_noise(torch.zeros_like(noise), noise, 91)
    g = torch.Generator(device="cuda").manual_seed(92)
    x = 1.5 - noise - width * torch.rand((rows, vocab), generator=g, device="cuda")
    run_sample(x, F32, 91)
    run_sample((x + 1e4)[:, 1:], F32, 93)


@pytest.mark.parametrize("rows", [2, 400])
def test_sample_masks_of_the_lowest_value(rows):
    """Rows of the type's lowest value, whose rank bound leaves the float range, alone and with live logits."""
    for dt, low in ((F16, -65504.0), (BF16, -3.3895313892515355e38), (F32, -3.4028234663852886e38)):
        x = np.full((rows, 12295), low, np.float32)
        x[1::2, 5000:5010] = np.linspace(-2, 2, 10)
        x[1::2, 12294] = 1.0
        run_sample(to_dev(orc.to_bits(x, dt), dt), dt, 94)


LOWEST = {F16: -65504.0, BF16: -3.3895313892515355e38, F32: -3.4028234663852886e38}


@pytest.mark.parametrize("rows,vocab", [(3, 30001), (16, 30000), (400, 12295)])
@pytest.mark.parametrize("dt", [F16, BF16, F32])
def test_sample_masked_slices(rows, vocab, dt):
    """Rows with slices that hold no live logit: -inf, -1e9 and lowest-value masks with a few live columns or none,
    a NaN or +inf somewhere, on the sliced kernels (three launches and one) and the row kernel."""
    rng = np.random.default_rng(rows)
    for low in (-np.inf, -1e9 if dt != F16 else -6e4, LOWEST[dt]):
        x = np.full((rows, vocab), low, np.float32)
        for r in range(rows):
            if r % 4:
                x[r, rng.integers(0, vocab, 5)] = rng.normal(0, 3, 5)
        x[0, vocab - 1] = (np.nan, np.inf, 1.0)[rows % 3]
        x[2, [7, vocab - 3]] = np.nan
        x[1, vocab // 2:] = -np.inf
        dev = to_dev(orc.to_bits(x, dt), dt)
        got = run_sample(dev, dt, 95)
        if rows < 384:
            ids = torch.empty(rows, dtype=torch.int64, device="cuda")
            ws = torch.zeros(ffi.sample_workspace_bytes(), dtype=torch.uint8, device="cuda")
            ffi.gumbel_sample_ws(dev, ids, ws, 0, 95)
            torch.cuda.synchronize()
            assert np.array_equal(ids.cpu().numpy(), got)


@pytest.mark.parametrize("rows", [16, 400])
def test_sample_where_the_noise_is_absorbed(rows):
    """Logits about the size (0x1.1p29) from which half the float spacing is more than any noise, on both sides of
    it, each row a few neighbouring floats of one size and sign: below it the noise still decides between them."""
    rng = np.random.default_rng(5)
    size = np.float32(2.0) ** rng.uniform(26, 33, (rows, 1)).astype(np.float32)
    size[:8, 0] = [2.0 ** 28, 2.0 ** 29, 570425344.0, np.nextafter(np.float32(570425344.0), 0), 2.0 ** 30, 1e9, 2.0 ** 31, 6e8]
    x = size.view(np.uint32) + rng.integers(-2, 3, (rows, 10250)).astype(np.uint32)
    x = x.astype(np.uint32).view(np.float32) * np.where(np.arange(rows) % 2, 1.0, -1.0)[:, None].astype(np.float32)
    run_sample(to_dev(np.ascontiguousarray(x), F32), F32, 96)


@pytest.mark.parametrize("rows", [16, 64])
def test_masked_draws_take_no_longer_than_live_ones(rows):
    """A top-k mask leaves most slices of a row without a live logit; they need no noise (us per draw of 151936 f32
    logits; with every masked candidate evaluated one by one, 20.3 against 9.3 at 16 rows and 27 against 14.3 at
    64).  The factor is for the clock."""
    live = dev_normal((rows, 151936), 0, 3, F32, 97)
    keep = torch.topk(live, 50, dim=1).indices
    ids = torch.empty(rows, dtype=torch.int64, device="cuda")
    us = {None: graph_us(lambda: ffi.gumbel_sample(live, ids, 0, 3))}
    for low in (-math.inf, -1e9, LOWEST[F32]):
        x = torch.full_like(live, low).scatter_(1, keep, live.gather(1, keep))
        us[low] = graph_us(lambda: ffi.gumbel_sample(x, ids, 0, 3))
    x = live.clone()
    x[:, 1000] = math.nan
    us["nan"] = graph_us(lambda: ffi.gumbel_sample(x, ids, 0, 3))
    assert max(us.values()) < 1.25 * us[None], us


@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("vocab", [1, 2048, 10240, 12289, 30001])
def test_sample_slice_lengths(chunks, vocab):
    """Every slice length, whole and cut short by the row's end, aligned rows and rows off by one element, and a last
    slice of one element."""
    from exl3r import _lib
    with _lib.tuned() as lib:
        lib.exl3r_tune_sample_slice(chunks)
        for dt in (F16, F32):
            x = dev_normal((5, vocab + 1), 0, 3, dt, 98)
            run_sample(x[:, :vocab].contiguous(), dt, 99)
            run_sample(x[:, 1:], dt, 99)
            run_sample(x, dt, 99, max(1, vocab - 4))


def test_fewer_rows_take_no_longer():
    """The slices follow the work of the whole draw: 15 rows (15.4 us in slices of 2048 logits) against 16 (9.3 in
    longer ones), and few rows of a small vocabulary against as many of a large one."""
    ids = torch.empty(16, dtype=torch.int64, device="cuda")
    x = dev_normal((16, 151936), 0, 3, F32, 100)
    few, many = (graph_us(lambda: ffi.gumbel_sample(x[:n], ids[:n], 0, 3)) for n in (15, 16))
    assert few < 1.15 * many, (few, many)


def test_rank_error_over_every_uniform():
    """The draw is exact as long as the hardware's log2 keeps the ranked noise within its bound of the exact noise,
    for every one of the 2^23 values of u."""
    from exl3r import _lib
    out = torch.full((2,), math.nan, device="cuda")
    _lib.check(_lib.load_tune().exl3r_tune_gumbel_rank_error(out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    err, bound = out.tolist()
    print(f"largest error {err:.3e}, bound {bound:.1e}")
    assert 0.0 < err < bound / 2
