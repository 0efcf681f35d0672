"""Decode of one or two sequences cut into up to 32 parts per head, against the
oracle: lengths around the lines of the shortest-chunk rule (an eighth of the
head, 160 KB of rows, 1/32 of the head), all row tiles, with and without the
append."""
import pytest

import nne_testlib as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("append", [True, False])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (16, 2, 128), (4, 4, 64), (2, 1, 256), (40, 2, 64)])
@pytest.mark.parametrize("lens", [[1279], [1281], [5121], [70, 9000]])
def test_long_heads_on_few_workgroups(nne, cuda, hq, hkv, d, lens, append):
    T.decode_vs_oracle(nne, cuda, len(lens), hq, hkv, d, lens, append, sum(lens) + d, "long heads")
