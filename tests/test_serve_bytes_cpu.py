"""The server's account of a scene that gives device memory back when it joins
its batch (its own sort buffers)."""
from __future__ import annotations

from mpm_amd.serve import Server
from tests.test_serve_cpu import Clock, FakeBackend, FakeBatch, FakeSolver, _req


class GivingSolver(FakeSolver):
    bytes = 1000

    def stats(self):
        return {"device_bytes": self.bytes, "cfl": 0.0}


class GivingBatch(FakeBatch):
    server, seen = None, []

    def add(self, s):
        super().add(s)
        s.bytes = 700

    def step(self, k):
        super().step(k)
        self.seen.append((len(self.members), self.server.used))


class GivingBackend(FakeBackend):
    def create_solver(self, desc, particles):
        return GivingSolver(desc, particles, self.log)

    def create_batch(self, interp, transfer):
        return GivingBatch((interp, transfer), self.clock, self.log)


def test_members_are_measured_after_they_joined():
    c = Clock()
    srv = Server(backend=GivingBackend(c), clock=c, sleep=c.sleep, build_threads=0)
    GivingBatch.server, GivingBatch.seen = srv, []
    rep = srv.run([_req(i, 0.0, 1000, 20) for i in range(3)])
    assert rep.failed == 0 and rep.completed == 3
    assert GivingBatch.seen and all(used == 700 * members for members, used in GivingBatch.seen)
