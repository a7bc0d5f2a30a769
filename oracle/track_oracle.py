"""FP64 CPU oracle for the tracking loop on a drift line with space charge.

TEST INFRASTRUCTURE ONLY.  This module is the oracle for
``ocelot_amd.track_drift``: it restates the loop of the reference's
``track()`` (ocelot/cpbd/track.py:462-485) on a line of drifts and markers,
with the navigator's split of each step into element sections
(ocelot/cpbd/navi.py:406-434), the first-order drift map of each section
(sc_oracle.drift), the space-charge kicks of the processes due at that step
(sc_oracle.apply) and the envelope after the step (envelope_oracle).  Which
process kicks at which step, and with which z_step, is the navigator's
scheduling (navi.py:343-398); it is taken as input, as the reference's
recorded schedule.  Only ``tests/`` may import it.

Pinned by golden vectors written by the reference's own track() on a
four-drift line (tests/golden/make_golden_track.py): the sections reproduce
the reference's particles bit for bit, and the Twiss list to rounding.
"""
import numpy as np

from oracle import envelope_oracle as eo
from oracle import sc_oracle as orc


class DriftLine:
    """Element lengths of a line (markers have length 0) and the navigator
    position state: z0, the current element and the sum of the lengths
    before it (navi.py:130-132)."""

    def __init__(self, lengths):
        self.lengths = [float(v) for v in lengths]
        self.z0 = 0.0
        self.n_elem = 0
        self.sum_lengths = 0.0

    @staticmethod
    def section_length(l, start, dl):
        """Length of the drift map built for a section of dl starting at
        start inside an element of length l (optic_element.py:361-402): the
        whole element when the section starts at its entrance and spans it,
        the rest of the element (l - start) when the section reaches its end,
        dl otherwise."""
        if start < 1e-10 and np.isclose(dl, l):
            return l
        if start + dl > l or np.isclose(start + dl, l):
            return l - start
        return dl

    def sections(self, dz):
        """Drift lengths the navigator maps a step of dz into, crossing
        element ends with a 1e-10 tolerance (navi.py:406-434); updates the
        position state as the navigator does."""
        out = []
        n = len(self.lengths)
        i = self.n_elem
        z1 = self.z0 + dz
        L = self.sum_lengths + self.lengths[i]
        while z1 + 1e-10 > L:
            dl = L - self.z0
            out.append(self.section_length(self.lengths[i], self.z0 + self.lengths[i] - L, dl))
            self.z0 = L
            dz -= dl
            if i >= n - 1:
                break
            i += 1
            L += self.lengths[i]
        if abs(dz) > 1e-10:
            out.append(self.section_length(self.lengths[i], self.z0 + self.lengths[i] - L, dz))
        self.z0 += dz
        self.sum_lengths = L - self.lengths[i]
        self.n_elem = i
        return out


def track_line(r, q, E, lengths, nav_dz, kicks, bounds=None):
    """track() on a drift line: for each navigator step of length nav_dz[k],
    the drift sections, then every kick scheduled at that step (``kicks[k]``:
    a list of (z_step, nmesh)), then the envelope.  r (6, n) is updated in
    place.  Returns the list of envelope dictionaries with "s" (cumulative
    step length, track.py:481-483)."""
    line = DriftLine(lengths)
    tws = [dict(eo.get_envelope(r, q, E, bounds=bounds), s=0.0)]
    s = 0.0
    for k, dz in enumerate(nav_dz):
        for dl in line.sections(float(dz)):
            orc.drift(r, dl, E)
        for zstep, nmesh in kicks[k]:
            orc.apply(r, q, E, zstep, nmesh)
        s += float(dz)
        tws.append(dict(eo.get_envelope(r, q, E, bounds=bounds), s=s))
    return tws
