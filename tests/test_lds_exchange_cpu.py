"""Where lanes of one wave read LDS rows that other lanes of it wrote, the source keeps the order:
a wave_lds_exchange() stands between the writes and the reads."""

from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "animaxs_amd" / "csrc"


# (file, start of the region, write, read): the write and the read occur in the region.
@pytest.mark.parametrize("name,start,write,read", [
    ("attention.hip", "void qk_prologue_d128_kernel", "lds[8 * i + (sub ^ i)] =", "= lds[8 * sub + (i ^ sub)]"),
    ("attention_short.hip", "load_chunk(0);", "put_chunk(kend);", "norm_chunk(kend);"),
    ("attention_short.hip", "load_chunk(0);", "put_row(qr,", "norm_row(qr,"),
    ("attention_short.hip", "for (int ch = 0;", "put_chunk(left", "norm_chunk(left"),
])
def test_exchange_between_write_and_read(name, start, write, read):
    src = (CSRC / name).read_text()
    src = src[src.index(start):]
    between = src[src.index(write):src.index(read)]
    assert "wave_lds_exchange();" in between
