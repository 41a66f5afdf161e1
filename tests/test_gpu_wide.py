"""GPU parity of the pair kernel's matrix-instruction mode (multipliers above
2^22, codewords above 32 bits): whole and partial column tiles, every number of
rows a lane, codewords up to 64 bits, alone, in batches and as server jobs."""
import pytest

import coding_reliability_amd as cra
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("rows", [2, 4, 8, 16])
@pytest.mark.parametrize("A", [(1 << 22) + 1, 58659 * 4097, (1 << 32) - 1, (1 << 32) + 1, (1 << 40) + 7,
                               (1 << 51) - 1, 0x5555555555555])
def test_wide_codes_against_oracle(ctx, A, rows):
    # row blocks of 128 .. 1024 words; 1 to 31 columns past the last tile of 32
    for N in [64 * rows, 64 * rows + 1, 64 * rows + 31, 128 * rows + 33, 192 * rows + 17, 4096, 4999]:
        if (N - 1) * A >> 64 or (N - 1) * A < 1 << 32:
            continue
        for chunk in (1, 3):
            raw, _ = ctx.an_pairs(A, N, rows_per_lane=rows, chunk_blocks=chunk)
            assert raw == O.an_pairs_raw(A, N, len(raw)), (N, chunk)


def test_every_mode_in_one_batch(ctx):
    codes = [(58659, 1000), ((1 << 52) - 5, 4095), (58659 * 4097, 3001), ((1 << 21) + 1, 5000), (61, 2049),
             (0xFFFFFFFFFFFF, 2500)]
    rows, _ = ctx.an_batch(codes)
    for (A, N), raw in zip(codes, rows):
        assert raw == O.an_pairs_raw(A, N, len(raw)), (A, N)


def test_wide_job_beside_a_narrow_one(ctx):
    stride = 4097
    with cra.Server(ctx) as srv:
        a = srv.submit(cra.JOB_AN_GRID, 26, A=58659, stride=stride)
        b = srv.submit(cra.JOB_AN_EXHAUSTIVE, 13, A=61)
        srv.wait(a)
        srv.wait(b)
        wide, narrow = srv.result(a)[0], srv.result(b)[0]
    assert wide == O.an_pairs_raw(58659 * stride, ((1 << 26) + stride - 1) // stride, len(wide))
    assert narrow == O.an_pairs_raw(61, 1 << 13, len(narrow))
