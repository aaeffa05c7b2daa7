"""Replay of the launches a forward or backward pass makes.

A pass of one (stage, micro-batch) launches the same kernels on the same stage-owned buffers in every batch.  It is recorded
while it is issued for the first time (:class:`hip.Plan`) and issued by one native call from then on.  The call skips the
layer code, and with it every check of an operand, so a plan stands for operands of one *form* only: what the checks look at,
all but the address.  Addresses are filled in at each launch; an operand of another form goes through the layer code again
and is recorded, or refused there, like a first one.
"""
from . import hip


def form(t):
    """What the checks and the choice of a kernel can see of an operand."""
    return None if t is None else (t.shape, t.dtype, t.stride(), t.device, t.data_ptr() & 15)


def _ranges(tensors):
    return [(t.data_ptr(), t.data_ptr() + hip.extent_bytes(t)) for t in tensors]


def _apart(ranges, others=()):
    """Whether none of ``ranges`` meets another one or one of ``others``."""
    meets = lambda a, b: a[0] < b[1] and b[0] < a[1]
    return not any(meets(a, b) for i, a in enumerate(ranges) for b in ranges[:i] + list(others))


class Replay:
    VARIANTS = 4     # forms remembered per (kind, stage, micro-batch)

    def __init__(self, module):
        self.module = module
        self.plans = {}      # (kind, stage, micro-batch) -> {form of the call: (plan, which operand or what it returns)}

    def run(self, slot, ctx, operands, variant, layers, step, issue):
        """``issue()``, or the replay of its launches.  ``operands``: the tensors (or None) the pass is given, which may be others
        in every call; everything else it touches belongs to the stage or to ``ctx``.  ``variant``: what else the pass depends
        on.  ``layers``: the pair (a, b) of the stage's layers it runs."""
        plans = self.plans.setdefault(slot, {})
        key = (ctx, variant) + tuple(map(form, operands))
        given = [t for t in operands if t is not None]
        known = plans.get(key)
        if known is not None:
            plan, at, out = known
            plan.launch(step, ctx.stream, given)
            return out if at is None else operands[at]
        own = self.module.pass_buffers(slot[1], slot[2], layers) + ctx.buffers()
        if not _apart(_ranges(given), _ranges(own)):
            return issue()     # a pointer into both would be taken for the operand's
        ctx.dropout_keys = {}
        try:
            with hip.Plan.record() as plan:
                out = issue()
            keys = ctx.dropout_keys
        finally:
            ctx.dropout_keys = None
        try:
            plan.dropout(keys)
            plan.operands(given)
        except hip.HipKernelError:      # the pass has run; it just cannot be replayed
            return out
        while len(plans) >= self.VARIANTS:
            del plans[next(iter(plans))]
        at = next((i for i, t in enumerate(operands) if t is out and t is not None), None)
        plans[key] = (plan, at, out if at is None else None)
        return out
