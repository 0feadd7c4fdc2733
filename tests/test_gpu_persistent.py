"""Persistent launches (one cooperative launch for many ticks, the block's states in registers,
the spike ring exchanged device-coherently across XCDs, a grid barrier between ticks) against
the CPU oracle and against one launch per tick: identical dumps, bit for bit."""
import numpy as np
import pytest

import nets
from atlas_hip import engine, models, protocol
from atlas_hip.executor import HipExecutor
from atlas_hip.models import hex_array
from atlas_hip.results import write_events, write_results
from oracle import oracle

pytestmark = pytest.mark.gpu


def run(doc, mode, monkeypatch, plain=False, **kwargs):
    monkeypatch.setenv("ATLAS_HIP_PERSISTENT", ("plain" if plain else "1") if mode == "persistent" else "0")
    with HipExecutor(doc, device=0, **kwargs) as ex:
        result = ex.run()
        assert result["hip_runtime"]["launch_mode"] == mode
        return write_results(ex.document, result), write_events(ex.document, result), result


def test_tenth_scale_persistent_equals_oracle_and_per_tick(monkeypatch):
    """Config 3's network at 100k neurons (in-degree 1000, 1e8 synapses), 150 ticks."""
    print("case: persistent scaled CUBA 100k x 1000, 150 ticks", flush=True)
    doc = models.cuba_network(100_000, indegree=1000, delay_ticks=1, steps=150, weight_scale=0.0116)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events > 1_000_000
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert dump == expected.results and events == expected.events
    assert result["hip_runtime"]["launches"] == 1
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch, lift_recording_budget=True)
    assert tick_dump == dump and tick_events == events


def test_plain_persistent_launches_equal_cooperative_ones(monkeypatch):
    """The same kernel issued as ordinary launches (the grid fits the device at once by its
    occupancy) gives the oracle's dump, over launches of 40 ticks."""
    print("case: plain persistent launches, scaled CUBA 100k x 1000, 120 ticks", flush=True)
    monkeypatch.setattr(engine, "PERSISTENT_TICKS", 40)
    doc = models.cuba_network(100_000, indegree=1000, delay_ticks=1, steps=120, weight_scale=0.0116)
    expected = oracle.run(doc, lift_recording_budget=True)
    dump, events, result = run(doc, "persistent", monkeypatch, plain=True, lift_recording_budget=True)
    assert result["hip_runtime"]["launches"] == 3
    assert dump == expected.results and events == expected.events


def test_persistent_run_split_over_launches(monkeypatch):
    """A run of 150 ticks in launches of 37 ticks (the states pass through memory between them)."""
    print("case: persistent scaled CUBA 100k x 1000, launches of 37 ticks", flush=True)
    monkeypatch.setattr(engine, "PERSISTENT_TICKS", 37)
    doc = models.cuba_network(100_000, indegree=1000, delay_ticks=1, steps=150, weight_scale=0.0116)
    expected = oracle.run(doc, lift_recording_budget=True)
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert result["hip_runtime"]["launches"] == 5
    assert dump == expected.results and events == expected.events


def test_persistent_synchronous_burst(monkeypatch):
    """Every neuron starts above threshold: all 100k fire at tick 0 (256 per block, so the ring
    records' first 7 ids and the id lists are both read), then 1e8 events arrive at tick 1."""
    print("case: persistent burst 100k x 1000, 30 ticks", flush=True)
    doc = models.cuba_network(100_000, indegree=1000, delay_ticks=1, steps=30, weight_scale=0.0116)
    doc["instance"]["populations"][0]["initial_state"]["v"] = hex_array(np.full(100_000, -0.0495), "f32")
    protocol.seal(doc)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events >= 100_000 * 1000
    dump, events, _ = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert dump == expected.results and events == expected.events


def test_large_blocks_with_long_segments_equal_oracle_and_per_tick(monkeypatch):
    """280,000 neurons forced into 4096-neuron blocks of 1024 work-items, one workgroup per CU (the
    executor would take 2048); at in-degree 1000 a (source, block) segment holds 14.6 targets on
    average, so about 40% exceed a slot's 15 inline targets and are read from the row table.  100
    ticks: the persistent launch equals the oracle and one launch per tick."""
    print("case: persistent 280k x 1000 in 4096-neuron blocks, 100 ticks", flush=True)
    doc = models.cuba_network(280_000, indegree=1000, delay_ticks=1, steps=100, weight_scale=0.0116)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events > 1_000_000
    shape = engine.Shape(4096, 1024, 2, 11)
    monkeypatch.setenv("ATLAS_HIP_PERSISTENT", "1")
    with HipExecutor(doc, device=0, shape=shape, lift_recording_budget=True) as ex:
        assert ex.plan.shape == shape and ex.plan.total_blocks == 69
        result = ex.run()
        assert result["hip_runtime"]["launch_mode"] == "persistent"
        dump, events = write_results(ex.document, result), write_events(ex.document, result)
    assert dump == expected.results and events == expected.events
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch, lift_recording_budget=True)
    assert tick_dump == dump and tick_events == events


def test_large_block_burst_reads_long_segments(monkeypatch):
    """100k neurons forced into 25 blocks of 4096 (in-degree 1000: about 41 targets per segment,
    nearly every slot read from the row table), every neuron firing at tick 0 so that 1e8
    events arrive at tick 1, over 20 ticks: equal to the oracle."""
    print("case: persistent burst 100k x 1000 in 4096-neuron blocks, 20 ticks", flush=True)
    monkeypatch.setattr(engine, "PERSISTENT_MIN_BLOCKS", 16)
    doc = models.cuba_network(100_000, indegree=1000, delay_ticks=1, steps=20, weight_scale=0.0116)
    doc["instance"]["populations"][0]["initial_state"]["v"] = hex_array(np.full(100_000, -0.0495), "f32")
    protocol.seal(doc)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events >= 100_000 * 1000
    dump, events, _ = run(doc, "persistent", monkeypatch, lift_recording_budget=True,
                          shape=engine.Shape(4096, 1024, 2, 11))
    assert dump == expected.results and events == expected.events


@pytest.mark.parametrize("model,ticks", [("cuba", 10_000), ("cobahh", 10_000)])
def test_delay_zero_persistent_equals_oracle_and_per_tick(monkeypatch, model, ticks):
    """Configs 1 and 2 (4000 neurons, Bernoulli p = 0.02, delay 0; 16 blocks of 256): each tick's
    deliveries follow its own publication and barrier inside the persistent launch.  CUBA's two
    pathways share the population as source range, so each fired source loads one slot per
    pathway.  Equal to the oracle and to one launch per tick (which delivers the previous tick
    first and the last tick in an epilogue)."""
    print(f"case: persistent delay 0, {model} 4000, {ticks} ticks", flush=True)
    doc = (models.cuba_network(4000, steps=ticks) if model == "cuba" else models.cobahh_network(4000, steps=ticks))
    # COBAHH in the oracle's libm mode: for this network its dump equals the shared-math mode's
    # (test_gpu_parity.py compares the device with the shared-math mode over the same ticks)
    expected = oracle.run(doc)
    dump, events, result = run(doc, "persistent", monkeypatch)
    assert result["hip_runtime"]["launches"] == 1
    assert dump == expected.results and events == expected.events
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch)
    assert tick_dump == dump and tick_events == events


def test_full_size_persistent_equals_per_tick(monkeypatch):
    """Config 3 at its full size (1M neurons, 1e9 synapses), 60 ticks: the persistent launch and one
    launch per tick give the same raster, states and event counts."""
    print("case: persistent scaled CUBA 1M x 1000, 60 ticks", flush=True)
    doc = models.cuba_network(1_000_000, indegree=1000, delay_ticks=1, steps=60, weight_scale=0.0116)
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True, verify_envelope=False)
    assert len(result["populations"][0]["spike_ticks"]) > 10_000
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch, lift_recording_budget=True,
                                    verify_envelope=False)
    assert tick_dump == dump and tick_events == events


def test_persistent_longer_delay(monkeypatch):
    """Delay 3: each tick's deliveries wait for the spikes of tick - 3 only, so workgroups drift up
    to three ticks apart and the ring holds 2 d + 2 = 8 ticks."""
    print("case: persistent scaled CUBA 100k x 1000, delay 3, 200 ticks", flush=True)
    doc = models.cuba_network(100_000, indegree=1000, delay_ticks=3, steps=200, weight_scale=0.0116)
    expected = oracle.run(doc, lift_recording_budget=True)
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert dump == expected.results and events == expected.events


@pytest.mark.parametrize("delay,ticks,per_launch", [(0, 12_000, 12_000), (1, 20_000, 10_000)])
def test_runs_past_the_stamp_period_equal_oracle_and_per_tick(monkeypatch, delay, ticks, per_launch):
    """Ring words carry a 12-bit stamp that repeats every lcm(R, 4095) ticks: 4095 for delay 0's ring
    of 3 (here inside one launch of 12,000 ticks), 16,380 for delay 1's ring of 4 (here across two
    launches of 10,000).  Each publication clears the words its slot's previous tick wrote past its
    own count, so no stale word can carry the stamp a reader waits for.  CUBA 4000 (Bernoulli
    p = 0.02): equal to the oracle and to one launch per tick."""
    print(f"case: persistent delay {delay}, CUBA 4000, {ticks} ticks in launches of {per_launch}", flush=True)
    monkeypatch.setattr(engine, "PERSISTENT_TICKS", per_launch)
    doc = models.cuba_network(4000, steps=ticks, delay_ticks=delay)
    expected = oracle.run(doc)
    dump, events, result = run(doc, "persistent", monkeypatch)
    assert result["hip_runtime"]["launches"] == -(-ticks // per_launch)
    assert dump == expected.results and events == expected.events
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch)
    assert tick_dump == dump and tick_events == events


WEIGHTED_SHAPE = engine.choose_shape(1_000_000, 1)   # 4096-neuron blocks of 1024 work-items


def weighted(n, steps, **kwargs):
    return models.cuba_network(n, indegree=1000, delay_ticks=1, steps=steps, weight_scale=0.0116, edge_weights=True,
                               **kwargs)


def test_weighted_split_loop_equals_oracle_and_per_tick(monkeypatch):
    """Config 3's network with a float32 weight per synapse at 100k neurons in 4096-neuron blocks
    (25 workgroups of the split loop, edge-keyed lists applied in key order): the oracle's dump over
    150 ticks in one launch and in launches of 37 ticks, and the same as one launch per tick (the
    ordered LDS path)."""
    print("case: weighted split loop 100k x 1000, 150 ticks", flush=True)
    doc = weighted(100_000, 150)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events > 1_000_000
    monkeypatch.setenv("ATLAS_HIP_PERSISTENT", "1")
    with HipExecutor(doc, device=0, lift_recording_budget=True, shape=WEIGHTED_SHAPE) as ex:
        assert ex.plan.populations[0].fused_edges and "EDGE_SLOTS = true" in ex.plan.source
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True, shape=WEIGHTED_SHAPE)
    assert result["hip_runtime"]["launches"] == 1
    assert dump == expected.results and events == expected.events
    monkeypatch.setattr(engine, "PERSISTENT_TICKS", 37)
    dump37, events37, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True, shape=WEIGHTED_SHAPE)
    assert result["hip_runtime"]["launches"] == 5
    assert dump37 == dump and events37 == events
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch, lift_recording_budget=True, shape=WEIGHTED_SHAPE)
    assert tick_dump == dump and tick_events == events


def test_weighted_split_loop_burst_replays_per_tick(monkeypatch):
    """Every neuron starts above threshold, so 1e8 weighted events arrive at tick 1, 4e6 per block:
    more than a block's edge lists hold.  The launch reports it and the run is replayed with one
    launch per tick, equal to the oracle."""
    print("case: weighted split loop burst 100k x 1000, 30 ticks", flush=True)
    doc = weighted(100_000, 30)
    doc["instance"]["populations"][0]["initial_state"]["v"] = hex_array(np.full(100_000, -0.0495), "f32")
    protocol.seal(doc)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events >= 100_000 * 1000
    monkeypatch.setenv("ATLAS_HIP_PERSISTENT", "1")
    with HipExecutor(doc, device=0, lift_recording_budget=True, shape=WEIGHTED_SHAPE) as ex:
        assert ex.launch_mode == "persistent"
        result = ex.run()
        assert ex.launch_mode == "per-tick"
        dump, events = write_results(ex.document, result), write_events(ex.document, result)
    assert dump == expected.results and events == expected.events


def test_weighted_full_size_split_loop_equals_per_tick(monkeypatch):
    """The weighted network at its full size (1M neurons, 1e9 synapses with their own weights), 60
    ticks: the split loop's edge lists and one launch per tick give the same dump."""
    print("case: weighted split loop 1M x 1000, 60 ticks", flush=True)
    doc = weighted(1_000_000, 60)
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True, verify_envelope=False)
    assert len(result["populations"][0]["spike_ticks"]) > 10_000
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch, lift_recording_budget=True, verify_envelope=False)
    assert tick_dump == dump and tick_events == events


@pytest.mark.parametrize("edge_weights,delay", [(False, 1), (False, 0), (True, 1)])
@pytest.mark.parametrize("indegree", [200, 260, 1100])
def test_segments_longer_than_a_slot_equal_oracle_and_per_tick(monkeypatch, indegree, edge_weights, delay):
    """4,200 neurons in 17 blocks of 256: (source, block) segments of 12, 16 and 65 targets on average, so
    lengths on both sides of a slot's inline targets (15, or 12 with a weight per synapse) and of a
    wave's 64 lanes, which share a longer segment's edges.  The persistent launches (the split loop
    at delay 1, by counters or edge buckets) and one launch per tick equal the oracle."""
    print(f"case: long segments, in-degree {indegree}, weights {edge_weights}, delay {delay}", flush=True)
    doc = models.cuba_network(4200, indegree=indegree, delay_ticks=delay, steps=400, weight_scale=11.6 / indegree,
                              edge_weights=edge_weights)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.synaptic_events > 50_000
    dump, events, _ = run(doc, "persistent", monkeypatch, lift_recording_budget=True,
                          shape=engine.Shape(256, 256, 4, 10))
    assert dump == expected.results and events == expected.events
    tick_dump, tick_events, _ = run(doc, "per-tick", monkeypatch, lift_recording_budget=True)
    assert tick_dump == dump and tick_events == events


@pytest.mark.parametrize("n,edge_weights", [(300, False), (300, True), (16_384, False), (16_385, True), (98_305, False),
                                            (98_305, True), (262_145, True), (524_289, False)])
def test_fitted_shapes_equal_the_oracle(monkeypatch, n, edge_weights):
    """Networks on both sides of the sizes where the executor's launch shape changes (2 blocks of 256;
    64 of 256; 33 of 512; 97 of 1024; 129 of 2048; 171 of 3072, ragged last blocks), with counted
    events and with a float32 weight per synapse: persistent, equal to the oracle."""
    print(f"case: fitted shape, {n} neurons, weights {edge_weights}", flush=True)
    doc = models.cuba_network(n, indegree=30, delay_ticks=1, steps=150, weight_scale=11.6 / 30,
                              edge_weights=edge_weights)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.spike_count > n // 20
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert dump == expected.results and events == expected.events
    assert result["hip_runtime"]["launches"] == 1


@pytest.mark.parametrize("doc", [
    models.delta_lif_network(300, indegree=20, steps=600),                       # 2 blocks, delays 2 and 1, late reset
    models.delta_lif_network(16_500, indegree=60, steps=300),                    # 33 blocks of 512
    models.delta_lif_network(4000, indegree=50, steps=400, delays=(1, 12), dtype="f64"),
    models.poisson_network(700, 1300, indegree=40, steps=800, delay_ticks=0),
    models.poisson_network(17_000, 300, indegree=300, steps=300, delay_ticks=1),  # 34 + 1 blocks of 512
    models.poisson_network(300, 17_000, indegree=30, steps=300, delay_ticks=5),   # 1 + 34 blocks of 512
    models.cuba_network(1024, p=0.05, steps=600)], ids=lambda doc: "")
def test_split_loop_of_several_groups_and_populations_equals_the_oracle(monkeypatch, doc):
    """The split loop over several counting groups of different delays, resets after the deliveries, a
    population that reads no spikes but waits for its readers, and delay 0: equal to the oracle in one
    launch and in launches of 37 ticks."""
    sizes = [pop["count"] for pop in doc["definition"]["populations"]]
    print(f"case: split loop, populations {sizes}", flush=True)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.spike_count > 100
    dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert dump == expected.results and events == expected.events
    assert result["hip_runtime"]["launches"] == 1
    monkeypatch.setattr(engine, "PERSISTENT_TICKS", 37)
    dump, events, _ = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
    assert dump == expected.results and events == expected.events


W = 0.1e-3   # V per event
SPLIT_GRAPHS = {   # population sizes, (source, target, delay, in-degree, weight), populations reset after the deliveries
    "three groups": ([700], [(0, 0, 1, 20, W), (0, 0, 5, 20, -W), (0, 0, 2, 20, W)], ()),
    "three groups, late reset": ([700], [(0, 0, 5, 20, W), (0, 0, 1, 20, -W), (0, 0, 2, 20, W)], (0,)),
    "five groups of 512-neuron blocks": ([9001], [(0, 0, d, 10, W * s) for d, s in zip((3, 1, 2, 1, 7), (1, -1, 1, 1, -1))], ()),
    "two populations reading each other": ([600, 900], [(0, 1, 2, 20, W), (1, 0, 5, 20, -W), (0, 0, 1, 20, W)], ()),
    "chain of three": ([300, 700, 513], [(0, 1, 1, 20, W), (1, 2, 4, 20, W)], ()),
    "cycle of three": ([300, 700, 513], [(0, 1, 1, 20, W), (1, 2, 4, 20, W), (2, 0, 6, 20, -W)], ()),
    "delay 0 beside others": ([300, 700], [(0, 1, 0, 20, W), (1, 0, 3, 20, -W), (1, 1, 0, 20, W)], ()),
    "delay 0 into a chain": ([300, 700, 513], [(0, 1, 0, 20, W), (1, 2, 0, 20, W), (0, 2, 7, 20, -W)], ()),
    "late reset of a population that others read": ([300, 700, 513], [(0, 1, 2, 20, W), (1, 1, 1, 20, -W), (1, 2, 3, 20, W)],
                                                    (1,)),
    "four coupled populations": ([300] * 4, [(i, j, 1 + (i + 2 * j) % 5, 10, W) for i in range(4) for j in range(4)], (2,))}


@pytest.mark.parametrize("name", SPLIT_GRAPHS)
def test_split_loop_over_population_graphs_equals_the_oracle(monkeypatch, name):
    """Populations that read each other, chains, cycles, three and more groups, delay 0 beside longer ones
    and resets after the deliveries in read populations, 700 ticks: the split loop equals the oracle in one
    launch and in launches of 37 ticks."""
    counts, paths, late = SPLIT_GRAPHS[name]
    print(f"case: split loop, {name}", flush=True)
    doc = nets.population_graph(counts, paths, steps=700, late=late)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.spike_count > sum(counts) // 2
    for ticks in (engine.PERSISTENT_TICKS, 37):
        monkeypatch.setattr(engine, "PERSISTENT_TICKS", ticks)
        dump, events, result = run(doc, "persistent", monkeypatch, lift_recording_budget=True)
        assert result["hip_runtime"]["launches"] == -(-700 // min(700, ticks))
        assert dump == expected.results and events == expected.events


def test_counters_past_the_lds_keep_one_launch_per_tick(monkeypatch):
    """600,000 neurons in six groups, whose counters pass the split loop's LDS: accepted, one launch per
    tick, equal to the oracle."""
    print("case: 600k neurons in six groups, 40 ticks", flush=True)
    doc = nets.population_graph([600_000], [(0, 0, 1 + k % 2, 2, W) for k in range(6)], steps=40)
    expected = oracle.run(doc, lift_recording_budget=True)
    assert expected.spike_count > 1000
    monkeypatch.setenv("ATLAS_HIP_PERSISTENT", "1")
    with HipExecutor(doc, device=0, lift_recording_budget=True) as ex:
        result = ex.run()
        assert result["hip_runtime"]["launch_mode"] == "per-tick"
        assert write_results(ex.document, result) == expected.results


@pytest.mark.parametrize("n,p,delay", [(64, 0.3, 0), (65, 0.3, 0), (1000, 0.05, 1), (2500, 0.03, 0)])
def test_sliced_update_equals_the_oracle(monkeypatch, n, p, delay):
    """COBAHH in blocks of 64 neurons whose update four replicas share: one block, a last block of one
    neuron, both orders of a tick; equal to the oracle in one launch and in launches of 37 ticks."""
    print(f"case: sliced COBAHH {n}, p {p}, delay {delay}", flush=True)
    doc = models.cobahh_network(n, p=p, steps=600, delay_ticks=delay)
    expected = oracle.run(doc)
    assert expected.spike_count > 30
    dump, events, result = run(doc, "persistent", monkeypatch)
    assert dump == expected.results and events == expected.events
    monkeypatch.setattr(engine, "PERSISTENT_TICKS", 37)
    dump, events, _ = run(doc, "persistent", monkeypatch)
    assert dump == expected.results and events == expected.events
