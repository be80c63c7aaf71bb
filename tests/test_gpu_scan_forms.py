"""The margin-filtered scan in each of its forms -- one, two or four neurons per lane, rows spread over sixteen
lanes or over quads -- at the edges of its rounds, chunks, slices and wavefronts, bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from helpers import dense_case
from oracle import capi
from test_gpu_parity import _adversarial_dense

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _check(x, w, p):
    import snntc_amd as snn
    ref_out, ref_k, _, _ = capi.fc_forward_dev(x, w, p, want_aux=True)
    out, _, _, ck = snn.snnfc(t(x), t(w), p, return_aux=True)
    out2 = snn.snnfc(t(x), t(w), p)
    torch.cuda.synchronize()
    assert np.array_equal(ck.cpu().numpy(), ref_k), "causal-set sizes differ"
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref_out.view(np.uint32)), "y / 1/S not bit-exact"
    assert torch.equal(out, out2)


SIZES = [
    (20011, 31, 64), (20011, 33, 63), (12007, 72, 128),     # 64-column slices, four neurons: below, above, between rounds
    (9001, 7, 50), (9001, 8, 50), (9001, 9, 50), (9001, 1, 40),          # rows of less than a chunk, one, one and a bit
    (6007, 650, 96), (3001, 785, 101),                      # 32-column slices: quads, and a ragged last slice
    (6007, 1301, 37), (700, 2305, 66),                      # 16-column slices
    (1500, 4600, 9), (40, 4601, 23),                        # 8-column slices, many wavefronts and few
    (1100, 400, 200), (300, 500, 70),                       # two neurons and one
]


@pytest.mark.parametrize("law", ["baseline", "initial", "small"])   # by the largest weight: either, the smallest weight sum tracked, bounded
@pytest.mark.parametrize("B,I,J", SIZES)
def test_scan_forms(B, I, J, law):
    """A tenth of the inputs (and all of every fiftieth row) never spiked, so rows of one wavefront differ in length."""
    from snntc_amd.layers import init_weight
    x, w, p, _ = dense_case(B + I, B, I, J, True, "baseline")
    if law == "initial":
        np.random.seed(B + I)
        w = init_weight(I, J, 1.0)
    elif law == "small":
        w = (0.12 + 0.01 * np.random.default_rng(J).standard_normal(w.shape)).astype(np.float32)
    rng = np.random.default_rng(I)
    x[rng.random(x.shape) < 0.1] = 1e5
    x[::50] = 2e5
    _check(x, w, p)


@pytest.mark.parametrize("B,I,J", [(13312, 4, 64), (13313, 4, 64), (7606, 7, 40), (700, 7, 261), (1000, 6, 33), (4096, 3, 32), (4097, 3, 32), (5, 2, 10),
                                   (49152, 1, 70), (49153, 1, 70), (1, 1, 1)])
@pytest.mark.parametrize("bias", [True, False])
def test_scans_of_less_than_a_chunk(B, I, J, bias):
    """Both sides of the line between weights in LDS and weights from memory; some rows silent in part or as a whole."""
    x, w, p, _ = dense_case(B + I + J, B, I, J, bias, "baseline")
    x[np.random.default_rng(I).random(x.shape) < 0.1] = 1e5
    x[::7] = 2e5
    _check(x, w, p)


# Launches that leave a SIMD a wavefront or two: rounds of twelve chunks (rows of sixteen lanes) and of eight (quads)
LONE_SIZES = [
    (700, 7, 64), (700, 95, 64), (700, 96, 64), (700, 97, 64), (700, 201, 63),          # 64-column slices, one neuron per lane
    (900, 96, 20), (900, 193, 20), (1200, 95, 10), (1200, 192, 16), (1200, 104, 11),    # 32 and 16 columns, rows of a wavefront in pairs and fours
    (1300, 127, 8), (1300, 128, 8), (1300, 192, 7), (1300, 259, 8), (40, 2689, 16),     # 8 columns: below and from the line on, several slices
    (6000, 288, 64), (6000, 299, 50), (2100, 700, 96), (512, 1345, 250),                # two neurons: 64, 32 and 16 columns
    (1536, 200, 130), (3300, 300, 96),                                                  # several turns, the last one partial
]


@pytest.mark.parametrize("law", ["baseline", "initial"])
@pytest.mark.parametrize("B,I,J", LONE_SIZES)
def test_scan_forms_of_small_launches(B, I, J, law):
    from snntc_amd.layers import init_weight
    x, w, p, _ = dense_case(B + I + J, B, I, J, True, "baseline")
    if law == "initial":
        np.random.seed(B + I)
        w = init_weight(I, J, 1.0)
    rng = np.random.default_rng(I)
    x[rng.random(x.shape) < 0.1] = 1e5
    x[::50] = 2e5
    x[7::50, I // 2:] = 1e5                                  # and rows that end early
    _check(x, w, p)


# Rows long enough to be tested a round of four chunks at a time at first, either side of that line, and slices of 64 columns that leave
# room for the row entries of sixteen wavefronts (up to 576 inputs) and that do not; other widths.
LONG_SIZES = [(12003, 399, 64), (12003, 400, 64), (12003, 431, 50), (12011, 576, 64), (12011, 577, 63), (12007, 608, 64), (12007, 609, 64),
              (12005, 624, 64), (12005, 625, 64), (12005, 638, 41), (9001, 700, 32), (5003, 1537, 16), (2603, 3001, 24), (1207, 4700, 16)]


# Two workgroups of four wavefronts to a CU, four neurons per lane: room for row entries in both (up to 304 inputs), and none
SHARED_SIZES = [(80, 289, 6400), (80, 304, 6400), (80, 305, 6400), (80, 319, 6400)]


@pytest.mark.parametrize("law", ["spread", "jump"])
@pytest.mark.parametrize("B,I,J", LONG_SIZES + SHARED_SIZES)
def test_scans_by_rounds(B, I, J, law):
    """`jump`: the times stand close together, then leap, so that a round fails that the one before it did not announce."""
    x, w, p, _ = dense_case(B + I + J, B, I, J, True, "baseline")
    rng = np.random.default_rng(I + J)
    if law == "jump":
        x = np.where(rng.random(x.shape) < rng.uniform(0.1, 0.9, (B, 1)), 1 + 0.3 * rng.random(x.shape), 3 + 0.2 * rng.random(x.shape)).astype(np.float32)
    x[1::3] = np.where(rng.random(x[1::3].shape) < 0.1, np.float32(1e5), x[1::3])
    x[::50] = 2e5
    x[7::50, I // 2:] = 1e5
    _check(x, w, p)


# The most inputs whose slice of 64, 32, 16 and 8 columns fits in LDS, with the bias row in memory, and one more
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("B,I,J", [(5003, 639, 64), (40, 639, 200), (2603, 1279, 40), (33, 1279, 100), (1207, 2559, 24), (49, 2559, 40), (605, 5118, 9), (9, 5118, 20), (9, 5119, 20)])
def test_widest_slices(B, I, J, bias):
    x, w, p, _ = dense_case(B + I + J, B, I, J, bias, "baseline")
    x[1::3] = np.where(np.random.default_rng(I).random(x[1::3].shape) < 0.1, np.float32(1e5), x[1::3])
    _check(x, w, p)


# Few wavefronts with rows of slices of eight columns, long ones and those of up to eight neurons from 1280 inputs on: whole turns of eight chunks
# and a chunk, an input more or less, and rows that end early.
@pytest.mark.parametrize("law", ["spread", "jump"])
@pytest.mark.parametrize("B,I,J", [(9, 2560, 64), (17, 2623, 40), (24, 2561, 64), (49, 3001, 70), (20, 4607, 33), (100, 4608, 200),
                                   (600, 1279, 8), (600, 1280, 8), (1000, 1343, 5), (300, 1345, 7), (700, 2047, 6)])
def test_long_rows_of_few_wavefronts(B, I, J, law):
    x, w, p, _ = dense_case(B + I + J, B, I, J, True, "baseline")
    rng = np.random.default_rng(I + J)
    if law == "jump":
        x = np.where(rng.random(x.shape) < rng.uniform(0.1, 0.9, (B, 1)), 1 + 0.3 * rng.random(x.shape), 3 + 0.2 * rng.random(x.shape)).astype(np.float32)
    x[1::3] = np.where(rng.random(x[1::3].shape) < 0.1, np.float32(1e5), x[1::3])
    x[-2, I // 2:] = 1e5
    x[-1] = 2e5
    _check(x, w, p)


# Launches whose workgroups order their own rows: one and two rows per item, networks of 512 and 1024, several slices
SORTING_SIZES = [(1, 784, 800), (1, 128, 30), (1, 129, 33), (3, 300, 20), (5, 511, 16), (6, 512, 40), (7, 513, 10), (5, 1023, 16), (2, 1024, 100),
                 (255, 800, 10), (1, 512, 1000), (100, 200, 64)]


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("B,I,J", SORTING_SIZES)
def test_scans_that_order_their_rows(B, I, J, ties):
    x, w, p, _ = dense_case(B + I + J, B, I, J, True, "baseline")
    rng = np.random.default_rng(I + J)
    if ties:
        x = (np.round(x * 16) / 16).astype(np.float32)
        x[:, ::7] = -0.0
        x[:, 3::7] = 0.0
    x[rng.random(x.shape) < 0.1] = 1e5
    x[-1, I // 3:] = 1e5
    x[B // 2, :] = 2e5
    _check(x, w, p)


@pytest.mark.parametrize("kind,B,I,J", [("randn", 700, 190, 64), ("ties", 900, 200, 25), ("negative", 1200, 175, 16),
                                        ("bias_fires", 1300, 200, 8), ("late", 700, 330, 64), ("sparse", 6000, 290, 64)])
def test_small_launches_off_the_common_path(kind, B, I, J):
    x, w = _adversarial_dense(kind, 3, B, I, J)
    _check(x, w, capi.fc_params(1.0))


@pytest.mark.parametrize("kind,B,I,J", [("randn", 20000, 90, 64), ("ties", 12000, 100, 61), ("negative", 9000, 75, 64),
                                        ("bias_fires", 9000, 131, 64), ("late", 9000, 330, 32), ("sparse", 4000, 700, 40)])
@pytest.mark.parametrize("small", [False, True])             # weights as they are, or scaled so that the smallest weight sum is bounded
def test_four_neuron_lanes_off_the_common_path(kind, B, I, J, small):
    x, w = _adversarial_dense(kind, 3, B, I, J)
    if small:
        w = (w * (0.19 / np.abs(w).max())).astype(np.float32)
    _check(x, w, capi.fc_params(1.0))


def test_scans_that_miss_their_close_by_a_rounding():
    """Among 1.5 million scans about a dozen pass their closing time unnoticed (the sums round the wrong way): they are
    left with a positive weight sum, not fired, and must be carried to the end of their rows, where practically all
    of them stay silent."""
    x, w, p, _ = dense_case(5, 24000, 600, 64, True, "baseline")
    _check(x, w, p)
