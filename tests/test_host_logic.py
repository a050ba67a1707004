"""Host functions of the library on the CPU, called from small C++ programs."""
import host_cpp


def test_batch_frame_key_covers_workgroup_setting(tmp_path):
    """traverse_blocks 0 and 4 per CU launch different grids: a frame captured
    under one is not replayed under the other."""
    host_cpp.run("batch_key", tmp_path)


def test_workgroup_setting_holds_for_every_launch(tmp_path):
    """traverse_blocks is the grid of a step and the most that a walk launches."""
    host_cpp.run("detect_grids", tmp_path)
