"""Buffer arguments that share memory, for the DOT4 products: a call whose
outputs overlap its activations never takes the one-launch (direct) GEMM, so
it reaches the split launches (up to 64 vectors) and the dense GEMM (more) at
any shape."""
import numpy as np


class At:
    """A place within a device array, as an operator's buffer argument."""

    def __init__(self, array, offset):
        self.array, self.ptr = array, type(array.ptr)(array.ptr.value + offset)


def copying_product(ctx, call, dm, act, rows, vectors, blocks, stride, fill=0.0):
    """call(ctx, matrix, activations, outputs, rows, vectors, blocks, stride)
    with the activations starting at the last four outputs: every chunk of
    vectors has been read before those are written. Returns the outputs
    [vectors][stride], the padding of the last row as `fill`."""
    act = np.ascontiguousarray(act).view(np.uint8).ravel()
    end = ((vectors - 1) * stride + rows) * 4
    host = np.concatenate([np.full((end - 16) // 4, fill, np.float32).view(np.uint8), act])
    both = ctx.array(host)
    call(ctx, dm, At(both, end - 16), both, rows, vectors, blocks, stride)
    out = np.full(vectors * stride, fill, np.float32)
    out[:end // 4] = both.download()[:end].view(np.float32)
    return out.reshape(vectors, stride)
