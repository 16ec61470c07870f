"""The tuner's cache belongs to a build of the library: a choice timed with other
kernels is not taken.  No device."""
import hashlib
import json

from eagleimp_amd import tune

from test_tune_host import _Engine, _Targets


def test_choice_of_other_kernels_is_not_taken(tmp_path, monkeypatch):
    monkeypatch.setattr(tune, "CACHE", str(tmp_path / "tune.json"))
    tg, batches = _Targets(300, 10000), (128, 256)
    # an entry as kept for the same panel, K, window and shapes by a library with
    # other kernels
    vs = tune.candidates(10000)
    sig = json.dumps([_Engine.Nad, _Engine.Ncorr, _Engine.M, 10000, 1000, list(batches),
                      [(v["threads"], v["chunks_per_wave"]) for v in vs]])
    key = hashlib.sha1(sig.encode()).hexdigest()[:16]
    (tmp_path / "tune.json").write_text(json.dumps({key: dict(variant=4, batch=128)}))
    eng = _Engine()
    best = tune.tune(eng, tg, range(300), batches=batches)
    assert not best["cached"] and best["variant"] == 3 and eng.submits > 0
    # and one of this library is, until the library changes
    assert tune.tune(_Engine(), tg, range(300), batches=batches)["cached"]
    other = tmp_path / "lib.so"
    other.write_bytes(b"another build")
    monkeypatch.setattr(tune, "LIB_PATH", str(other))
    assert not tune.tune(_Engine(), tg, range(300), batches=batches)["cached"]


def test_automatic_stays_on_where_it_starts_from_the_choice(tmp_path, monkeypatch):
    """The automatic choice starts from the smallest shape that holds K (2 at
    K = 10,000) and takes one with more threads for few targets: a tuned engine
    keeps that where the tuner picks the same shape, from the cache too."""
    monkeypatch.setattr(tune, "CACHE", str(tmp_path / "tune.json"))
    tg = _Targets(300, 10000)
    for per, variant, on in (({2: 1.0, 3: 2.0}, 2, -1), ({2: 2.0, 4: 1.0}, 4, 4)):
        for use_cache in (False, True, True):
            eng = _Engine(per=per)
            best = tune.tune(eng, tg, range(300), batches=(128, 256) if on < 0 else (256,),
                             use_cache=use_cache)
            assert best["variant"] == variant and eng.variant == on
        assert best["cached"]
