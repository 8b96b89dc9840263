"""The training update's guards on its LDS use (csrc/sp_mlp_train.h) hold where
its row chunks fit the partial sums' array and fail beyond."""
import os
import re

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stochastic-parker_amd", "csrc",
                   "sp_mlp_train.h")


@pytest.mark.parametrize("parts,fits", [(16, True), (17, False), (32, False)])
def test_bias_chunks_fit_the_partial_sums(parts, fits):
    text = open(SRC).read()
    names = {k: int(v) for k, v in re.findall(r"constexpr int (k\w+) = (\d+);", text)}
    names["kColParts"] = parts
    used = re.findall(r"part\[2 \* (?:pt|\(t >> 5\)) \+ ", text)
    assert used                                    # chunk p stores into rows 2 p and 2 p + 1 of part
    holds = all(eval(c, {}, names) for c in re.findall(r"static_assert\((.*kColParts.*), \"", text))
    assert holds == (2 * parts <= names["kUpdateSplits"]) == fits
