"""What a delta-rule layer says of a step's portions: the same for a filled-up description whichever step of its shape it is."""
import pytest

from tokenizer_amd.engine.batch import filled_counts
from tokenizer_amd.parts.delta import portion_rows


@pytest.mark.parametrize("lengths, least", [([1] * 12, 0), ([300] + [1] * 15, 100), ([40], 13), ([200] * 7 + [1] * 30, 200), ([24] * 8, 16),
                                            ([2048], 682)])
def test_rows_of_a_portion(lengths, least):
    tokens, entries, _, _, single = filled_counts(lengths, [0] * len(lengths))
    portions = [n for n in lengths if n > 1]
    average = (tokens - sum(lengths) + sum(portions)) / max(1, len(portions))           # (rows that fill the step up lie behind the portions)
    assert least <= portion_rows(tokens, entries, single) <= max(average, 0)
