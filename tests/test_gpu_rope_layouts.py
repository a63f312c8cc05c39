"""GPU parity of the RoPE kernel's layouts for heads of 64, 128 and 256 with full and partial rotary widths, and of
its two forms: the one that gives every wave one item at most (a decode batch, a short prefill) and the one that
walks the items, in front of and behind the switch.  Sources: inv_freq, the table of angles, the q | g split and
the paged append, each against the oracle at its own tests' tolerance."""
import numpy as np
import pytest

import exl3r
from oracle import oracle as orc
from test_gpu_rope import run as run_rope
from test_gpu_rope_paged import layout, run as run_paged
from test_gpu_rope_qg import run as run_qg
from test_gpu_rope_table import run as run_table

pytestmark = pytest.mark.gpu

F16, BF16, F32 = orc.F16, orc.BF16, orc.F32
NEOX = exl3r.ROPE_NEOX
LAYOUTS = [(64, 64), (64, 16), (128, 128), (128, 32), (256, 256), (256, 64), (256, 240)]
TOKENS = [1, 3, 4000]     # 1, 3: one item per wave; 4000 of 21 heads: more items than resident waves


@pytest.mark.parametrize("hd,R", LAYOUTS)
@pytest.mark.parametrize("seq", TOKENS)
def test_inv_freq(hd, R, seq):
    pid = np.random.default_rng(hd + R).integers(0, 30000, (1, seq)).astype(np.int32)
    run_rope(1, seq, 18, 3, hd, R, NEOX, F16, position_ids=pid, seed=hd, out_of_place=True)
    run_rope(1, seq, 18, 3, hd, R, NEOX, BF16, nwt=F32, cb=1.0, position=17, seed=R)
    run_rope(1, seq, 5, 3, hd, R, NEOX, F16, norm=False, position=2, with_k=False, seed=R + 1)


@pytest.mark.parametrize("hd,R", [(64, 64), (64, 32), (128, 128), (128, 64), (256, 64)])
@pytest.mark.parametrize("bsz,seq", [(2, 1), (2, 2000)])
def test_angle_tables(hd, R, bsz, seq):
    tables = np.random.default_rng(hd).uniform(-500.0, 500.0, (bsz, seq, R // 2)).astype(np.float32)
    run_table(bsz, seq, 18, 3, hd, tables, NEOX, F16, seed=hd)
    pid = np.random.default_rng(R).integers(0, seq + 1, (bsz, seq)).astype(np.int32)     # seq: outside the table
    pid[0, 0] = seq
    run_table(bsz, seq, 18, 3, hd, tables[0], NEOX, BF16, nwt=BF16, position_ids=pid, seed=R, expect_err=1)


def test_angle_tables_gptj():
    for seq in (3, 4000):
        tables = np.random.default_rng(3).uniform(-500.0, 500.0, (seq, 32)).astype(np.float32)
        run_table(1, seq, 18, 3, 128, tables, exl3r.ROPE_GPTJ, F16, seed=4)


@pytest.mark.parametrize("hd,R", [(64, 64), (128, 64), (256, 64)])
@pytest.mark.parametrize("seq", TOKENS)
def test_query_gate_split(hd, R, seq):
    run_qg(1, seq, 18, 3, hd, R, NEOX, BF16, nwt=BF16, cb=1.0, position=5, seed=hd)


@pytest.mark.parametrize("hd,R", [(64, 64), (128, 128), (128, 64), (256, 64)])
@pytest.mark.parametrize("bsz,seq", [(37, 1), (2, 2000)])
def test_paged_append(hd, R, bsz, seq):
    pages, bt, sl = layout(bsz, seq, 256, 9, hd)
    run_paged(bsz, seq, 13, 3, hd, R, NEOX, F16, 256, pages, 9, sl, bt, with_out_k=False, seed=hd)
    sl[0] = 9 * 256 - seq + 1                          # the first sequence's last position is past its block table
    bt[-1, :] = pages + 1                              # the last sequence's pages are outside the pool
    run_paged(bsz, seq, 13, 3, hd, R, NEOX, BF16, 256, pages, 9, sl, bt, seed=R)
