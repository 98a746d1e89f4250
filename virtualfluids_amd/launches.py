"""Sequences of launches enqueued by the library (vf_run_launches).

A time step is a fixed list of launches. Enqueued one by one from Python each costs about 8 us of
host time, more than a small kernel takes; a HIP graph of the steps takes the host out of the
loop but costs 250-400 us to capture, twice that with its single-step tails, and about 10 us
between replays. The native loop enqueues a launch in 2.6 us, from the first step on: 66^3 cavity,
us per step over 100 steps, 16.9 with graphs captured in the run, 12.7 from the loop.
"""
from __future__ import annotations

import ctypes
import math

import torch

from . import capi


# Repeats of a list per native call. Signals are answered between the calls, so a long run can be
# interrupted; a call costs about 5 us, under 1 % of 256 steps of the shortest launch
_REPEATS = 256


class LaunchList:
    """The launches of a time step, to be enqueued `repeats` times on a stream. The entries point at
    the caller's parameter structs, which a run reads as they then are; the list keeps them
    (and the structs of the BC lists and interface cells) alive. Build it for one run of steps: it
    does not follow a lattice whose lists or buffers are replaced."""

    def __init__(self):
        self._entries = []
        self._array = None
        self._keep = []

    def _add(self, kind, level, **fields):
        e = capi.Launch()
        e.kind = kind
        e.level = ctypes.pointer(level)
        for name, value in fields.items():
            setattr(e, name, value)
        self._keep.append((level, fields))
        self._entries.append(e)
        self._array = None

    def collide(self, level, box: bool, template: int = capi.COLLISION_DEFAULT):
        self._add(capi.LAUNCH_BOX if box else capi.LAUNCH_INDICES, level, collisionTemplate=template)

    def collide_bounce_back(self, level, bounce_back, template: int = capi.COLLISION_DEFAULT):
        self._add(capi.LAUNCH_BOX_BOUNCE_BACK, level, collisionTemplate=template,
                  bounceBack=ctypes.pointer(bounce_back))

    def bc(self, level, fn_name: str, bc_struct):
        self._add(capi.LAUNCH_BC, level, bc=ctypes.cast(getattr(capi.load(), fn_name), ctypes.c_void_p),
                  list=ctypes.pointer(bc_struct))

    def bc_pair(self, level, fn_name: str, velocity_struct, noslip_struct):
        self._add(capi.LAUNCH_BC, level, pair=ctypes.cast(getattr(capi.load(), fn_name), ctypes.c_void_p),
                  list=ctypes.pointer(velocity_struct), list2=ctypes.pointer(noslip_struct))

    def post_groups(self, level, groups):
        """The post-collision launches (simulation.paired_launches)."""
        for fn, bcs in groups:
            if len(bcs) == 2:
                self.bc_pair(level, fn, *(bc.struct for _, bc in bcs))
            else:
                self.bc(level, fn, bcs[0][1].struct)

    def swap(self, level):
        self._add(capi.LAUNCH_SWAP, level)

    def _scale(self, kind, coarse, fine, cells):
        fields = {"fine": ctypes.pointer(fine), "cells": ctypes.pointer(cells.struct)}
        if cells.offsets is not None:
            fields["offsets"] = ctypes.pointer(cells.neigh)
        self._add(kind, coarse, **fields)

    def fine_to_coarse(self, coarse, fine, cells):
        if cells.n:
            self._scale(capi.LAUNCH_FINE_TO_COARSE, coarse, fine, cells)

    def coarse_to_fine(self, coarse, fine, cells):
        if cells.n:
            self._scale(capi.LAUNCH_COARSE_TO_FINE, coarse, fine, cells)

    def run(self, repeats: int, stream=None):
        """Enqueue the list `repeats` times (a fraction counts as a whole one) on `stream` (default: the
        current stream)."""
        from .lattice import stream_handle

        if repeats <= 0 or not self._entries:
            return
        if self._array is None:
            self._array = (capi.Launch * len(self._entries))(*self._entries)
        while repeats > 0:
            n = math.ceil(min(repeats, _REPEATS))
            capi.call("vf_run_launches", self._array, len(self._entries), n, stream_handle(stream))
            repeats -= n


class StepLaunches:
    """Time steps that work in place on fixed buffers: run(n, even) takes n steps from parity `even`
    and returns the parity after them; calling the object takes one. With `launches` (the step's
    LaunchList and the parameter struct whose isEvenTimestep is the step's parity) they are enqueued
    natively; otherwise step(even, stream) launches each. close() ends them."""

    def __init__(self, step, launches=None):
        self.step = step
        self.launches = launches
        self.enqueued = 0

    def run(self, n: int, even: bool) -> bool:
        if self.launches is not None:
            program, param = self.launches
            param.isEvenTimestep = 1 if even else 0
            program.run(n)
            self.enqueued += n
            return bool(param.isEvenTimestep)
        for _ in range(n):
            self.step(even, torch.cuda.current_stream())
            even = not even
        return even

    def __call__(self, even: bool):
        self.run(1, even)

    def close(self):
        """Wait for the steps, as Simulation.run does: a sweep of three or more native steps has
        returned when they are done. Inside a caller's capture there is nothing to wait for."""
        if self.enqueued >= 3 and not torch.cuda.is_current_stream_capturing():
            torch.cuda.current_stream().synchronize()
