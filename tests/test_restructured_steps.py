"""Steps the device code restructures for fewer dependent memory accesses, checked by brute force against the literal
sequence they replace (which follows the reference line by line). The whole-tick parity tests cover them again in
context."""


def test_move_cells_equals_remove_then_push(oracle):
    """grid_broadphase.cuh:44-84: removing the old block's cells one by one, then pushing the new block's, equals the
    one-pass move_cells, including the overflow count when the list is full."""
    for p in ((0, 0), (6, 2)):
        w = oracle.build_world(*p)
        assert oracle.check_move_cells(w, 12345 + p[0], 100000) == 0


def test_island_sort_in_a_register_equals_the_literal_sort(oracle):
    """simulation_island_manager.cuh:43-66 and the ascending sort before it, over active lists of 0 to 16 entries with
    every mix of keys, some with repeated entries."""
    assert oracle.check_island_sort(99, 2000000) == 0


def test_broadphase_in_two_steps_equals_the_literal_swaps(oracle):
    """axis_sweep.cuh:49-127, grid_broadphase.cuh:68-84: updates that keep an axis's order written in place and the rest
    put off equal the swaps made one by one, bit for bit, through moves that reorder edges, add and remove pairs and move
    the cell blocks (also of several bodies at once)."""
    for p in ((0, 0), (6, 2)):
        w = oracle.build_world(*p)
        states = oracle.sample_arenas(w, 1, 7, 4)
        for k in range(4):
            assert oracle.check_sweep(w, states[k].copy(), 77 + k, 20000) == 0
