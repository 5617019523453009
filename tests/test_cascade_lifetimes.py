"""Host buffers of a cascade call outlive the wait for its streams: an object
at the top of star_cascade waits when the call returns or throws, and what is
declared after it is gone by then.  So every vector that a copy of the stream
reads or writes has to be declared before it (read from the source: a copy that
fails half way cannot be had on purpose)."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), '..', 'emustack_amd', 'csrc', 'cascade.hip')


def test_vectors_in_flight_are_declared_before_the_wait():
    with open(SRC) as f:
        text = f.read()
    body = text[text.index('void star_cascade('):]
    body = body[:body.index('\n}\n')]
    wait = body.index('} upl{')
    names = set(re.findall(r'hipMemcpyAsync\([^;]*?(\w+)\.data\(\)', body))
    assert len(names) >= 3
    for name in sorted(names):
        declared = re.search(r'std::vector<\w+>[^;]*\b%s\b' % name, body).start()
        assert declared < wait, name
