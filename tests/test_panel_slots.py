"""The LDS slots that the wavefronts of k_panel_reg exchange their pivot
candidates through, replayed on the host: a column step posts to one of two
buffers, passes one barrier and reads the same buffer, so the next step's posts
must go to the other one unless a barrier comes in between.  The buffer's
expression and the instantiations are taken from the kernel's source."""
import os
import re

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), '..', 'emustack_amd', 'csrc', 'kernels_lu.hip')
NB = 32  # columns of a panel


def _source():
    with open(SRC) as f:
        text = f.read()
    body = text[text.index('void k_panel_reg('):text.index('__global__', text.index('void k_panel_reg('))]
    expr = re.search(r'\bpb = ([^;]*);', body).group(1)
    inst = {tuple(int(x) for x in m) for m in re.findall(r'EMU_PANEL\((\d+), (\d+), (\d+)\)', text)}
    return expr, sorted(inst)


@pytest.mark.parametrize('nw,rpt,cw', _source()[1])
def test_successive_steps_post_to_different_buffers(nw, rpt, cw):
    expr = _source()[0]
    for w in range(1, NB + 1):
        for c0 in range(0, w, cw):
            last = None  # buffer that waves may still be reading; a chunk ends with barriers
            for j0 in (0, cw // 2):
                for jj in range(cw // 2):
                    if j0 + jj >= min(cw, w - c0):
                        continue
                    pb = eval(expr, {}, dict(j0=j0, jj=jj, c0=c0, k0=0, k=c0 + j0 + jj))
                    assert nw == 1 or pb != last, (w, c0 + j0 + jj)
                    assert pb in (0, 1)
                    last = pb


def test_instantiations_are_found():
    assert len(_source()[1]) >= 7
