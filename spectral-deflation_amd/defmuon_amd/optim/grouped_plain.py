"""Grouped launches for the plain polar arms ("ns5", "polarexpress").

The reference's plain Muon step calls the factorizer once per parameter
(muon.py:361-386): at GPT-2 sizes that is a stream of small, occupancy-bound
launches.  Muon's own step takes buckets of parameters (Muon.PLAIN_BUCKET bytes)
with one library launch per (matrix shape, dtype, orientation) of a bucket;
`install()` lifts the limit, the way deflation_cutoff.install()
(deflation_cutoff.py:46-112) changes Muon's behaviour from outside.  Every
parameter's update is that of its own factorizer call
(Muon._muon_step_plain_grouped).  The deflated arms batch by shape already.
"""

_INSTALLED = [False]


def install():
    """One bucket per parameter group for every Muon instance (idempotent)."""
    if _INSTALLED[0]:
        return
    _INSTALLED[0] = True
    from defmuon_amd.optim.muon import Muon
    Muon.GROUPED_PLAIN = True


def uninstall():
    """Back to buckets of Muon.PLAIN_BUCKET bytes."""
    from defmuon_amd.optim.muon import Muon
    Muon.GROUPED_PLAIN = False
    _INSTALLED[0] = False
