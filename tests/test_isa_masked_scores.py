"""CPU-side check of the code generated for gfx950: the short form masks the scores of a ragged end, a masked range or a causal
diagonal with comparisons and selects.  A change of the execution mask per score, and with it 17 instructions instead of 4,
took 0.5 to 1 us of a small call, whose only step this is."""
import os
import re

import pytest

from mojodiffusion_amd import _lib
from test_isa_tile_copies import OBJDUMP, _functions


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no LLVM tools")
def test_no_branch_per_masked_score(tmp_path):
    seen = 0
    for symbol, code in _functions(_lib.LIB_PATH, tmp_path).items():
        # <D, variant, key runs, Q in the kernel, bias> = <.., .., .., false, false>: 16 scores of a lane and step with fp16 P.V, 32 with e4m3
        if re.match(r"_ZN4sage22sage_attn_short_kernelILi\d+ELi[01]ELi[48]ELb0ELb0EEE", symbol) and code:
            seen += 1
            assert sum(op == "s_and_saveexec_b64" for _, op, _, _ in code) < 8, symbol
    assert seen == 10
