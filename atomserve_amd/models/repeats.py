"""Layers like the ones before them, launched from a list.

A step that is not replayed as a graph (a prompt's portion, a mixed step) is launched kernel by kernel, and between two
launches of 4 us stand some 9 us of Python: parts that choose kernels, wrappers that check every tensor.  For a layer
like one that has just run (equal specs, the same step) all of that comes out the same, so a stretch of one or a few
layers is run once with its calls written down (`kernels.lib.Launches`) and the calls are made again for every
further stretch, the weights' and caches' addresses replaced by that stretch's.  Nothing outlives the step.

What one stretch leaves for the next (the pending output of its last part) lies in two sets of buffers in turn: the ones that the
written-down stretch read and the ones that it wrote.
"""

import torch

from atomserve_amd.kernels import ops
from atomserve_amd.kernels.lib import Launches
from atomserve_amd.parts.base import DeltaSum, SplitSums
from atomserve_amd.parts.block import PreNormBlock, TwoNormsBlock
from atomserve_amd.parts.norm import PendingRMSNorm

MOST_LAYERS = 4  # of a stretch
# Steps of more tokens are left alone: their kernels take longer than the host, and the buffers that a stretch holds are larger
# (Qwen3-0.6B sizes, the smallest model: 1,024 tokens take the GPU as long as the host).
MOST_TOKENS = 1024


def _plain(block) -> bool:
    """Whether the layer is of a kind whose launches may be written down, with nothing put in place of its methods."""
    return type(block) in (PreNormBlock, TwoNormsBlock) and "forward" not in vars(block) and all(
        "forward" not in vars(part) for part in block.parts().values())  # fmt: skip


def stretches(plan, blocks) -> tuple:
    """(first run, layers of a stretch, stretches after it) that covers the most runs, or None: runs from the first one on
    repeat the ones before them with equal specs, all writing caches of their own."""
    runs, best = plan.run, None

    def alike(i, j) -> bool:
        a, b = runs[i], runs[j]
        return (not a.reenter and not b.reenter and a.writes and b.writes and plan.cache_id(i) == i and plan.cache_id(j) == j
                and a.layer != b.layer and type(blocks[a.layer]) is type(blocks[b.layer])
                and blocks[a.layer].spec == blocks[b.layer].spec and not blocks[a.layer].cache_request()
                and (blocks[a.layer].parts().keys() == blocks[b.layer].parts().keys()))  # fmt: skip

    def follows(i):
        """What the run before `i` is told of the norm that comes."""
        norm = blocks[runs[i].layer].first_norm() if i < len(runs) else None
        return None if norm is None else (type(norm), norm.spec)

    for period in range(1, MOST_LAYERS + 1):
        for first in range(1, len(runs) - 2 * period + 1):
            count = 0
            while True:
                at = first + (count + 1) * period
                if at + period > len(runs) or follows(at + period) != follows(first + period) or not all(
                        alike(first + k, at + k) for k in range(period)):  # fmt: skip
                    break
                count += 1
            if count and (best is None or count * period > best[1] * best[2]):
                best = (first, period, count)
    return best


def _view_parts(view, into: list) -> None:
    """What a cache view or a dict of views holds, in an order that equal kinds share: tensors, and numbers as they are."""
    if isinstance(view, dict):
        for name in sorted(view):
            _view_parts(view[name], into)
    elif view is not None:
        into.extend([getattr(view, name) for name in type(view).__slots__])


class _Own:
    """What belongs to a stretch and takes the place of the written-down one's: its layers' tensors (all of their parts'
    attributes that are tensors or `ops.Streamed`, a matrix and its copy), its caches and the gains of the norms that follow its
    layers (which their last products may prepare).

    Beside its address a launch carries types, shapes and layouts that the wrappers have checked for the written-down stretch
    alone, and gains may be stored in 32 bits in one layer and in 16 in another (a checkpoint says so tensor by tensor): every
    tensor that the launches read has to be of the same kind in every stretch, and what one stretch does without, all do."""

    def __init__(self, model, step, first: int, period: int):
        self.model, self.step, self.tensors = model, step, []
        # per layer: its class, its parts' attributes as (part, class, [(attribute, whether it has a copy)]) and those of the norm that follows
        self.layers = []
        for k in range(period):
            block, names = model.blocks[model.plan.run[first + k].layer], []
            for name, part in block.parts().items():
                wanted = [(attr, isinstance(v, ops.Streamed)) for attr, v in vars(part).items()
                          if v is None or isinstance(v, (torch.Tensor, ops.Streamed))]  # fmt: skip
                names.append((name, type(part), wanted))
            after = self.norm_after(first + k)
            self.layers.append((type(block), names, [attr for attr, v in vars(after).items() if v is None or isinstance(v, torch.Tensor)]
                                if after is not None else []))  # fmt: skip
        self.tensors = self.of(first)

    def norm_after(self, i: int):
        run = self.model.plan.run
        return self.model.blocks[run[i + 1].layer].first_norm() if i + 1 < len(run) else None

    def of(self, start: int):
        """Tensors, numbers of the caches and None, of the stretch that starts at run `start`; None where a layer is of another
        class, something stands in place of its methods, or a plain tensor for a matrix with a copy or the other way round."""
        model, plan, found = self.model, self.model.plan, []
        for i, (kind, names, gains) in enumerate(self.layers, start):
            block = model.blocks[plan.run[i].layer]
            if type(block) is not kind or "forward" in vars(block):
                return None
            parts = block.parts()
            for name, kind, wanted in names:
                have = vars(parts[name])
                if type(parts[name]) is not kind or "forward" in have:
                    return None
                for attr, streamed in wanted:
                    v = have.get(attr)
                    if streamed:
                        if type(v) is not ops.Streamed:
                            return None
                        found.append(v.rows)
                        found.append(v.wave)
                    else:
                        found.append(v)
            _view_parts(self.step.cache_view(plan.cache_id(i), True), found)
            if gains:
                have = vars(self.norm_after(i))
                found.extend([have.get(attr) for attr in gains])
        return found

    def addresses(self) -> list:
        return [v.data_ptr() if isinstance(v, torch.Tensor) else 0 for v in self.tensors]

    def read(self, places: list) -> None:
        """The places whose tensors the launches read."""
        at, self.met, self.alike = {}, [], []
        for i in places:
            v = self.tensors[i]
            if at.setdefault(id(v), i) == i:
                self.met.append((i, v, v.data_ptr(), v.dtype, v.shape, v.is_contiguous()))
            else:
                self.alike.append((i, at[id(v)]))  # one tensor under two names
        places = set(places)
        self.plain = [(i, v) for i, v in enumerate(self.tensors) if not isinstance(v, torch.Tensor)]
        self.unread = [i for i, v in enumerate(self.tensors) if isinstance(v, torch.Tensor) and i not in places]

    def targets(self, start: int):
        """The addresses of the stretch that starts at run `start` where the launches read them, or None if it is of another kind."""
        own = self.of(start)
        if own is None or len(own) != len(self.tensors):
            return None
        found = [0] * len(own)
        for i, source, address, dtype, shape, contiguous in self.met:
            v = own[i]
            if v is not source:  # what all layers of a step share is itself
                if v is None or v.dtype is not dtype or v.shape != shape or v.is_contiguous() != contiguous:
                    return None
                there = v.data_ptr()
                if (there - address) & 15:  # kernels are chosen by it
                    return None
                address = there
            found[i] = address
        for i, j in self.alike:
            if own[i] is not own[j]:
                return None
            found[i] = found[j]
        for i, v in self.plain:
            if own[i] is not v and (isinstance(own[i], torch.Tensor) or own[i] != v):
                return None
        for i in self.unread:
            if own[i] is None:
                return None
        return found


def _left(delta):
    """The tensors of a pending output, or None for a kind that is not handed on here."""
    if isinstance(delta, torch.Tensor):
        return [delta]
    if isinstance(delta, SplitSums):
        return [delta.sums]
    if type(delta) is PendingRMSNorm:
        return [delta.scaled, delta.ssq]
    if isinstance(delta, DeltaSum) and all(isinstance(p, torch.Tensor) for p in delta.parts):
        return list(delta.parts)
    return None


def run_again(model, made: Launches, step, before, after, first: int, period: int, count: int):
    """The `count` stretches after the one that starts at run `first`, whose launches `made` holds; before, after: the pending
    outputs that it took and gave.  Returns (runs done, the pending output); (0, after) if they are not its like."""
    taken, given = _left(before), _left(after)
    if not made.whole or taken is None or given is None or type(before) is not type(after) or \
            [(t.shape, t.dtype) for t in taken] != [(t.shape, t.dtype) for t in given]:  # fmt: skip
        return 0, after
    turns = [[t.data_ptr() for t in taken], [t.data_ptr() for t in given]]

    own = _Own(model, step, first, period)
    made.aim(own.addresses() + turns[0] + turns[1])
    own.read([i for i in made.met if i < len(own.tensors)])
    done = 0
    for _ in range(count):
        targets = own.targets(first + done + period)
        if targets is None:
            break
        targets += turns[1] + turns[0]
        if not made.fits(targets):
            break
        made.again(targets)
        turns.reverse()
        before, after = after, before
        done += period
    if done and type(after) is PendingRMSNorm:  # the norm that is pending is the next run's
        after = PendingRMSNorm(model.blocks[model.plan.run[first + period + done].layer].first_norm(), after.x, after.scaled, after.ssq)
    return done, after


def may_run_again(model, step, first: int, period: int) -> bool:
    """Whether the stretch that starts at run `first` is worth writing down in this step."""
    return (step.num_tokens <= MOST_TOKENS and not model.env.products.trials_pending()
            and not torch.cuda.is_current_stream_capturing()
            and all(_plain(block) and all(part.repeats(step) for part in block.parts().values())
                    for block in (model.blocks[model.plan.run[first + k].layer] for k in range(period))))  # fmt: skip
