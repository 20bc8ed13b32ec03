"""The NF4 quantizer's constant tables on the host."""

import torch

from causal_tuner.quant import nf4


def test_constant_tables_do_not_depend_on_the_default_device():
    """The tables kept per device are host values copied there: a default device in force on the
    first call (here meta, whose values cannot be copied; a GPU would compute them on the
    caller's stream) leaves no trace in them."""
    device = torch.device("cpu")
    nf4._device_tables.cache_clear()
    with torch.device("meta"):
        tables = nf4._device_tables(device)
    want = nf4.nf4_thresholds(), nf4.nf4_code(), nf4.dynamic_map()
    assert all(t.device == device and torch.equal(t, w) for t, w in zip(tables, want))
    assert nf4._device_tables(device) is tables
