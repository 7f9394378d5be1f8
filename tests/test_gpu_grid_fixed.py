"""The PME grid's fixed-point conversions (pgm_eval_grid_fixed).

The spread converts an atom's contributions A t3 + C u3 in a few instructions when charge, dipole and fractions allow
it, and in the general way otherwise.  What either gives is a whole number: over the admitted range they are equal bit for
bit.  An atom whose charge, dipole or position is not finite, or beyond the range, is not admitted: the fast conversion
would add the bit pattern of a NaN to the grid of all atoms.
"""

import numpy as np
import pytest

from pgmhip import engine as E

pytestmark = pytest.mark.gpu

LIMIT = {"double": 2.0**26, "mixed": 2.0**18}


@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_admitted_atoms(precision):
    lim = LIMIT[precision]
    plain = [0.4, 1.0, -2.0, 0.5, 0.0, 0.25, 1.0]
    rows, want = [plain], [1]
    for k in range(7):
        for bad in (np.nan, np.inf) + ((-np.inf, lim, -lim) if k < 4 else ()):
            rows.append(plain[:k] + [bad] + plain[k + 1 :])
            want.append(0)
    rows += [[lim - 8, 0, 0, 0, 1.0, 1.0, 1.0], [0, 0, -(lim - 8), 0, 1.0, 1.0, 1.0]]
    want += [1, 1]
    words = E.eval_grid_fixed(precision, rows, np.zeros(len(rows)))
    np.testing.assert_array_equal(words[:, 0], want)


@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_fast_conversion_gives_the_same_words(precision):
    rng = np.random.default_rng(4)
    mag = np.exp(rng.uniform(np.log(1e-20), np.log(LIMIT[precision]), 400000))
    unit = 2.0 ** -(24 if precision == "double" else 32)
    ties = (np.arange(-2000, 2000) + 0.5) * unit   # halfway between two words
    v = np.concatenate([mag, -mag, ties, [0.0, -0.0, LIMIT[precision] - 1.0, 1.0 - LIMIT[precision]]])
    if precision == "mixed":
        v = v.astype(np.float32).astype(np.float64)
    words = E.eval_grid_fixed(precision, np.zeros((len(v), 7)), v)
    np.testing.assert_array_equal(words[:, 3:], words[:, 1:3])
    np.testing.assert_array_equal(words[:, 1], np.rint(v / unit).astype(np.int64))
