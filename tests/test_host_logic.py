"""Host functions of the library on the CPU, called from small C++ programs."""
import host_cpp


def test_batch_frame_key_covers_workgroup_setting(tmp_path):
    """traverse_blocks 0 and 4 per CU launch different grids: a frame captured
    under one is not replayed under the other."""
    host_cpp.run("batch_key", tmp_path)


def test_workgroup_setting_holds_for_every_launch(tmp_path):
    """traverse_blocks is the grid of a step and the most that a walk launches."""
    host_cpp.run("detect_grids", tmp_path)


def test_overlapped_batch_query_leaves_room(tmp_path):
    """An overlapped batch frame's query launches as an overlapped scene's does: four
    workgroups a CU for a step, two for a walk."""
    host_cpp.run("overlap_grids", tmp_path)


def test_pair_sample_of_lists_that_follow_its_stride(tmp_path):
    """No bucket of the pair lists' sample sort outgrows LDS on lists whose order
    repeats at any distance."""
    host_cpp.run("pair_sample", tmp_path)


def test_walks_follow_the_fronts_that_a_check_has_read(tmp_path):
    """Steps guessed short that meet fronts far past the walks' limits are
    planned by those lengths from the next query on, until they fit the guess."""
    host_cpp.run("walk_plan", tmp_path)


def test_checks_do_not_spin_where_waits_block(tmp_path):
    """A program that chose blocking or yielding waits keeps its core while a check
    waits for the GPU."""
    host_cpp.run("check_wait", tmp_path)
