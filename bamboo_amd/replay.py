"""Replay of the launches a forward or backward pass makes.

A pass of one (stage, micro-batch) launches the same kernels on the same stage-owned buffers in every batch.  It is recorded
while it is issued for the first time (:class:`hip.Plan`) and issued by one native call from then on.  The call skips the
layer code, and with it every check of an operand and every look at a setting.  So

* a plan stands for operands of one *form*: what the checks look at, all but the address.  Addresses are filled in at each
  launch; an operand of another form goes through the layer code again and is recorded, or refused there, like a first one;
* the plans of a stage stand for one *state* of its layers: the attributes of each layer, its weights and the buffers, compared
  at every pass.  Another state drops them;
* only layers that say so are replayed (``launches_only``): a pass of any other layer is issued as always.
"""
from operator import is_

from . import hip


# what a class may define without saying anything about its passes
_HARMLESS = {"__init__", "__repr__", "__module__", "__qualname__", "__doc__", "__dict__", "__weakref__", "__annotations__", "__parameters__",
             "__orig_bases__", "init_params", "num_params", "flops_fwd"}


# what passes call on a layer (PipelineModule.pass_state has those of a given pass)
PASS_METHODS = ("forward", "backward", "rebuild", "grad_sink")


def _promises(kind):
    promised = False
    for cls in kind.__mro__[:-1]:
        own = vars(cls)
        if own.get("launches_only") is True:
            promised = True
            if any(getattr(own.get(m), "__module__", cls.__module__) != cls.__module__ for m in PASS_METHODS):
                return False
        elif not own.keys() <= _HARMLESS:
            return False
    return promised


def launches_only(layers):
    """Whether the passes of ``layers`` do nothing that a replay of their launches leaves out.  A class promises it for what it
    defines by ``launches_only = True`` of its own; a subclass without it may define how its parameters start
    (``_HARMLESS``) and no more, and nothing may be put over a method on the object or in place of one in the class."""
    kinds = set(map(type, layers))
    if not all(map(_promises, kinds)):
        return False
    names = {kind: set(dir(kind)) - {"__dict__"} for kind in kinds}
    return all(names[type(layer)].isdisjoint(vars(layer)) for layer in layers)


def form(t):
    """What the checks and the choice of a kernel can see of an operand."""
    return None if t is None else (t.shape, t.dtype, t.stride(), t.device, t.data_ptr() & 15)


def _apart(ranges, others):
    """Whether none of ``ranges`` meets one of ``others``."""
    for lo2, hi2 in others:
        for lo, hi in ranges:
            if lo < hi2 and lo2 < hi:
                return False
    return True


_NONE = {}


class Replay:
    VARIANTS = 4     # forms remembered per (kind, stage, micro-batch)

    def __init__(self, module, *stores):
        """``stores``: further dicts whose keys have the stage second, emptied with the plans when a stage's state changes."""
        self.module = module
        self.plans = {}      # (kind, stage, micro-batch) -> {form of the call: (plan, which operand or what it returns)}
        self._stores = stores
        # (stage, layers) -> (state that what is stored was recorded under, the memory passes use under it; None: not to be replayed)
        self._states = {}
        self._kinds = set()  # (kind, stage, layers) of the passes seen

    def forget(self):
        """Drop every plan, and with the states the references to what the passes used."""
        self.plans.clear()
        self._states.clear()
        self._kinds.clear()

    def settled(self, stage_id, ctx, layers):
        """Whether passes of these layers may be replayed; drops what was recorded under another state of theirs."""
        new = self.module.pass_state(stage_id, layers)
        new += ctx.pass_state()
        old, memory = self._states.get((stage_id, layers), (None, None))
        # identity: the list keeps every object alive, numbers and strings do not change, and dicts are in it with their values
        if old is not None and len(old) == len(new) and all(map(is_, old, new)):
            return memory is not None
        if old is not None:
            for store in (self.plans,) + self._stores:
                stale = [k for k in store if k[1] == stage_id]
                if stale and store is not self.plans:
                    ctx.stream.synchronize()     # captured graphs are destroyed here
                for k in stale:
                    del store[k]
        fit = self.module.passes_launch_only() and launches_only(self.module.func_buckets[stage_id][slice(*layers)])
        memory = list(map(hip.address_range, self.module.stage_memory(stage_id) + ctx.buffers())) if fit else None
        self._states[(stage_id, layers)] = (new, memory)
        return fit

    def _told_apart(self, slot, ctx, ranges, layers):
        """Whether a recorded pointer can belong to one operand only, and to nothing else that the pass uses."""
        if not all(_apart([r], ranges[:i]) for i, r in enumerate(ranges)):
            return False
        # (first against the stage's blocks of memory, then against what the pass itself has of them: one layer's input lies
        # in the same block as its output)
        return _apart(ranges, self._states[(slot[1], layers)][1]) or \
            _apart(ranges, map(hip.address_range, self.module.pass_buffers(slot[1], slot[2], layers) + ctx.buffers()))

    def run(self, slot, ctx, operands, variant, layers, step, issue):
        """``issue()``, or the replay of its launches.  ``operands``: the tensors (or None) the pass is given, which may be others
        in every call; everything else it touches belongs to the stage or to ``ctx``.  ``variant``: what else the pass depends
        on.  ``layers``: the pair (a, b) of the stage's layers it runs."""
        if not self.settled(slot[1], ctx, layers):
            return issue()
        key = (ctx, variant) + tuple(map(form, operands))
        given = [t for t in operands if t is not None]
        known = self.plans.get(slot, _NONE).get(key)
        if known is not None:
            plan, at, out = known
            plan.launch(step, ctx.stream, given)
            return out if at is None else operands[at]
        ranges = list(map(hip.address_range, given))
        if not self._told_apart(slot, ctx, ranges, layers):
            return issue()
        ctx.dropout_keys = {}
        try:
            with hip.Plan.record() as plan:
                out = issue()
            keys = ctx.dropout_keys
        finally:
            ctx.dropout_keys = None
        try:
            plan.dropout(keys)
            plan.operands(ranges)
        except hip.HipKernelError:      # the pass has run; it just cannot be replayed
            return out
        kind = (slot[0], slot[1], layers)
        if kind not in self._kinds:
            # a layer may make attributes of its own in its first pass: what was recorded in front of that is of no use
            self._kinds.add(kind)
            if not self.settled(slot[1], ctx, layers):
                return out
        plans = self.plans.setdefault(slot, {})
        while len(plans) >= self.VARIANTS:
            del plans[next(iter(plans))]
        at = next((i for i, t in enumerate(operands) if t is out and t is not None), None)
        plans[key] = (plan, at, out if at is None else None)
        return out
