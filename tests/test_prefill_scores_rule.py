"""Which kernel computes a prompt's DECODE router scores (host arithmetic in the library, no GPU): the one that was the
faster at the sizes on either side of each line. Times in us with 64 experts on an MI355X."""
import pytest

ANY, REGS, MFMA = 0, 1, 2

# hidden, tokens, us with any row path, us with the rows in registers (None: not for this hidden size), us on the MFMA
TIMES = [
    (256, 1, 2.85, 2.29, 5.98), (256, 769, 12.16, 4.69, 7.83), (256, 2048, 12.58, 7.41, 8.01),
    (256, 2049, 12.52, 8.06, 7.98), (256, 3001, 12.72, 10.09, 8.13),
    (512, 769, 19.31, 6.37, 9.83), (512, 1792, 19.68, 9.50, 9.98), (512, 1793, 19.65, 10.42, 9.96),
    (768, 769, 26.05, 7.57, 11.80), (768, 1792, 26.55, 11.43, 12.04), (768, 1793, 26.45, 12.53, 11.99),
    (1024, 769, 32.98, 13.58, 14.03), (1024, 1024, 33.03, 13.79, 14.08), (1024, 1536, 33.12, 19.04, 14.18),
    (1280, 256, 39.66, 7.14, 15.95), (1280, 768, 39.83, 13.90, 16.01), (1280, 769, 39.75, 16.83, 16.00),
    (1280, 3001, 40.17, 43.44, 16.64),
    (1536, 1, 7.00, None, 15.87), (1536, 2, 12.62, None, 16.52), (1536, 3, 18.06, None, 17.02),
    (1536, 1024, 46.98, None, 18.02),
    (1792, 2, 14.34, None, 18.49), (1792, 3, 20.70, None, 19.04),
    (2048, 1, 8.63, None, 19.83), (2048, 2, 15.88, None, 20.52), (2048, 3, 22.85, None, 21.06),
    (2048, 16, 59.10, None, 21.72),
]


@pytest.mark.parametrize("H,T,any_us,regs_us,mfma_us", TIMES)
def test_the_faster_kernel_is_taken(lib, H, T, any_us, regs_us, mfma_us):
    us = {ANY: any_us, REGS: regs_us, MFMA: mfma_us}
    fastest = min((k for k in us if us[k] is not None), key=lambda k: us[k])
    assert lib.load().dsh_pf_scores_kind(H, 64, T, 16) == fastest


@pytest.mark.parametrize("H", [256, 1280, 2048])
def test_single_rows_take_the_general_kernel(lib, H):
    """16 threads give 16 experts chunks of one row: the single-row path, which only one kernel has."""
    L = lib.load()
    for T in (1, 100, 3001):
        assert L.dsh_pf_scores_kind(H, 16, T, 16) == ANY
        assert L.dsh_pf_scores_kind(H, 16, T, 8) != ANY or (H > 1280 and T <= 2)
