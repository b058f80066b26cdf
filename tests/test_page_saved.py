"""A page whose escape stream is a view of a larger buffer, saved and loaded again."""
import io

import torch

from gaac_amd import Page


def test_a_saved_page_holds_the_stream_only():
    i32 = dict(dtype=torch.int32)
    room = torch.full((1 << 16,), 7, dtype=torch.uint8)
    page = Page(torch.zeros(1, 2048, dtype=torch.uint8), torch.zeros(1, 768, dtype=torch.uint8), torch.zeros(1, 16, **i32), torch.zeros(1, 16, **i32), room[:40],
                torch.tensor([0, 32], **i32), torch.zeros(1, 1, **i32), torch.zeros(1, 128, dtype=torch.uint8), torch.zeros(1, 128, dtype=torch.uint8), 1, 16, 1, "k")
    f = io.BytesIO()
    torch.save(page, f)
    assert len(f.getvalue()) < 1 << 15
    f.seek(0)
    again = torch.load(f, weights_only=False)
    assert torch.equal(again.ovf, page.ovf) and again.ovf.untyped_storage().nbytes() == 40 and again.nbytes == page.nbytes
    assert page.ovf.data_ptr() == room.data_ptr()      # the page itself is left as it was
