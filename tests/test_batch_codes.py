"""What the batched calls take as codes: pairs of integers, nothing else."""
import pytest

import coding_reliability_amd as cra


@pytest.mark.parametrize("codes", [[(61, 256, 7), (3, 16, 9)], [(61,), (3,)], [(61.5, 256)], [(61, 256.0)], ["61"]])
@pytest.mark.parametrize("call", ["autotune_batch", "an_batch", "batch_plan"])
def test_anything_but_integer_pairs_is_refused(call, codes):
    ctx = cra.Context.__new__(cra.Context)  # without a device: refused before it is asked for
    ctx._h = None
    with pytest.raises((TypeError, ValueError, AttributeError)):
        getattr(ctx, call)(codes)


def test_autotuner_takes_numpy_integers():
    import numpy as np
    ctx = cra.Context.__new__(cra.Context)
    ctx._h = None
    with pytest.raises(cra.CRError):  # the library's answer to no context
        ctx.autotune_batch(np.array([[61, 256], [3, 16]]))
