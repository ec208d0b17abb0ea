"""The tile that a contraction without one runs on (host rules of libdcc; no GPU calls), at launches that were
timed with every tile: the choice is one of those within 5 % of the best that was measured."""
import pytest

from distr_cc import _lib as L


def _map(*levels):
    """dcc_idxmap of (extent, stride) levels, outermost first."""
    lv = [(1, 0)] * (3 - len(levels)) + list(levels)
    return L.IdxMap(None, 0, lv[1][0], lv[2][0], lv[0][1], lv[1][1], lv[2][1])


def _tile(kind, rows, N, K, beta, am, ak, bk, bn, cm, cn, nbatch):
    return L._lib.dcc_contract_default_tile(kind, N, K, beta, 4096, am, ak, 8192, bk, bn, cm, cn, nbatch, rows)


# terms of z4 / t4 of (Q) at (nocc, nvir, blksize): rows, N, K, batches, maps of C, best tiles (times in us of the
# chosen ones against 64x128 or 128x64, which the area rule took)
Q_TERMS = [
    # nocc=10, nvir=24, blksize 4, 'abej,cdekli': 160 x 4000 x 24: 0: 1510, 4: 1510, 5: 2080, 6: 2187
    (160, 4000, 24, 208, (4, 10, 400000, 100000, 100), (160, 10, 10000, 1, 1000), (0, 4)),
    # nocc=16, nvir=8, blksize 2, 'dabeij,eclk': 1024 x 512 x 8: 0: 389, 4: 415, 6: 675
    (1024, 512, 8, 70, (4, 256, 65536, 262144, 256), (16, 16, 131072, 1, 16), (0,)),
    # nocc=15, nvir=8, blksize 6, 'cmkl,adbimj' (C contiguous along m): 4: 838, 5: 964, 0: 973
    (1350, 8100, 15, 12, (6, 225, 0, 303750, 1), (15, 15, 1822500, 3375, 225), (4,)),
    # nocc=15, nvir=8, blksize 6, 'dbej,aceikl' (C contiguous along n): 4: 693, 5: 708, 6: 713
    (90, 20250, 12, 72, (6, 15, 50625, 1822500, 225), (15, 225, 303750, 3375, 1), (4, 5, 6)),
]


@pytest.mark.parametrize("rows,N,K,nbatch,cm,cn,best", Q_TERMS)
def test_accumulated_short_k(rows, N, K, nbatch, cm, cn, best):
    m = lambda e1, e2, s0, s1, s2: L.IdxMap(None, 0, e1, e2, s0, s1, s2)
    am, ak, bk, bn = _map((rows, 1)), _map((K, rows)), _map((K, N)), _map((N, 1))
    assert _tile(0, rows, N, K, 1.0, am, ak, bk, bn, m(*cm), m(*cn), nbatch) in best
    # FP32, a product that is written only, and a longer K keep the shape of the area rule
    wide = _tile(0, rows, N, K, 0.0, am, ak, bk, bn, m(*cm), m(*cn), nbatch)
    assert wide == _tile(0, rows, N, 41, 1.0, am, ak, bk, bn, m(*cm), m(*cn), nbatch)


def test_few_outputs_stay_on_the_skinny_tiles():
    am, ak, bk, bn = _map((64, 1)), _map((8, 64)), _map((8, 64)), _map((64, 1))
    for kind in (0, 1):
        assert _tile(kind, 64, 64, 8, 1.0, am, ak, bk, bn, _map((64, 64)), _map((64, 1)), 1) >= 64
    assert _tile(9, 64, 64, 8, 1.0, am, ak, bk, bn, _map((64, 64)), _map((64, 1)), 1) == -1


# split-BF16x3 launches by how their operands load: rows, N, K, batches, inner extent of B's K, best tiles (times in
# us; the rule by areas alone took 8 or 9 for each of them but the last two)
BF16X3 = [
    # packed pairs, nvir = 50: 128x128 against 256x256, 804: 1123 and 842: 1398
    ("pairs", 2500, 14300, 2500, 1, 2500, (3,)),
    ("pairs", 2500, 14300, 2500, 1, 50, (3,)),
    # ring at nocc=10, nvir=90: 3402: 4572
    ("pairs", 900, 8100, 900, 55, 90, (3,)),
    # packed pairs of a short K against 156 rows: one pass over the long operand, 216: 328
    ("pairs", 156, 514500, 78, 1, 78, (8,)),
    # packed quads, 360 tiles of 256x256: 150: 218
    ("quads", 820, 11440, 832, 2, 832, (3,)),
    ("quads", 5460, 17160, 5504, 2, 5504, (8,)),
    # single words, nvir = 107: 31114: 47667; 1080 x 1080 x 102 over 1080 batches: 4607..4735
    ("single", 11449, 30602, 11449, 1, 11449, (8,)),
    ("single", 472, 472, 67, 472, 67, (3, 8)),
    # operands split in the tile: t3 -> W_vvvo at nocc=9, nvir=73: 671: 827, nocc=6, nvir=88: 231: 326
    ("unpacked", 47961, 73, 5913, 1, 73, (3, 9)),
    ("unpacked pairs", 46464, 88, 3168, 1, 88, (3,)),
    ("unpacked", 1440, 1, 14400, 144, 14400, (1,)),
]


@pytest.mark.parametrize("loads,rows,N,K,nbatch,ke,best", BF16X3)
def test_split_bf16x3(loads, rows, N, K, nbatch, ke, best):
    packed = not loads.startswith("unpacked")
    step = {"quads": 4, "pairs": 2, "unpacked pairs": 2}.get(loads, 1)
    assert K % step == 0 and N % step == 0
    pad = (8, 6, 5)[(step == 2) + 2 * (step == 1)]     # the row stride decides what an aligned vector can hold
    stride = -(-max(K, N) // 8) * 8 + pad
    am, ak = _map((rows, stride)), _map((K, 1))
    # B contiguous along K in runs of ke
    bk = _map((K // ke, stride * N), (ke, 1)) if ke < K else _map((K, 1))
    bn = _map((N, stride))
    assert _tile(3 if packed else 2, rows, N, K, 0.0, am, ak, bk, bn, _map((rows, N)), _map((N, 1)), nbatch) in best
