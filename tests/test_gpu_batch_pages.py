"""Volume sets defined before the pool: the page ids are unchecked then and cost no memory."""
import resource

import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import workloads as W
from hydrant_amd.hip import Context, batch_config

pytestmark = pytest.mark.gpu


def test_page_ids_beyond_any_pool(gpu_ctx):
    """A set whose pages no pool holds is taken while there is none, costs what its cells cost, and
    is refused at the launch; a set of pages that the later pool holds renders."""
    import torch

    wl = W.batched(sizes=(40,), n_views=2, res_choices=(33, 64), fmt=L.FMT_U8, bs=16, apron=1, seed=11)
    descs = wl.volume_descs()
    far = [dict(d, vaddr=np.where(np.asarray(d["vaddr"]) >= 0, 2 ** 31 - 2, -1).astype(np.int32)) for d in descs]
    ctx = Context(0)
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
    ctx.set_volumes(far)
    assert resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before < 1 << 20   # KiB: 1 GiB
    ctx.upload_pool(wl.fmt, wl.bs + 2 * wl.apron, wl.pool)
    ctx.set_tf(wl.tf)
    b = ctx.batch(wl.hip_views())
    with pytest.raises(Exception, match="names page"):
        b.render(batch_config(8, 4, 8, 1), wl.density, 0.0)
    b.close()
    images = []
    for late in (False, True):   # the same set before and after its pool
        ctx.close()
        ctx = Context(0)
        if late:
            ctx.set_volumes(descs)
        ctx.upload_pool(wl.fmt, wl.bs + 2 * wl.apron, wl.pool)
        if not late:
            ctx.set_volumes(descs)
        ctx.set_tf(wl.tf)
        b = ctx.batch(wl.hip_views())
        images.append(b.render(batch_config(8, 4, 8, 1), wl.density, 0.0)[0].clone())
        torch.cuda.synchronize()
        b.close()
    ctx.close()
    assert torch.equal(images[0], images[1])
