"""ctypes binding of the C-ABI in include/dynet_hip.h (libdynet_hip.so)."""
import ctypes as C
import os
import re
import subprocess

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libdynet_hip.so")
HEADER_PATH = os.path.join(os.path.dirname(_HERE), "include", "dynet_hip.h")
CSRC_DIR = os.path.join(_HERE, "csrc")

OK, ERR_INVALID_ARG, ERR_RUNTIME, ERR_OUT_OF_MEMORY, ERR_NO_DEVICE = range(5)
POOL_FXS, POOL_DEDFS, POOL_PS, POOL_SCS = range(4)
SCALAR_MINUSONE, SCALAR_ONE, SCALAR_ZERO = range(3)
OP_TANH, OP_LOGISTIC, OP_RECTIFY, OP_NEGATE, OP_IDENTITY = range(5)
LOGISTIC_PACKET, LOGISTIC_SCALAR = 0, 1
CWISE_SUM, CWISE_MULT, CWISE_QUOTIENT = range(3)
LN_STATIC_SCRATCH_BYTES = 4 << 20  # DYHIP_LN_STATIC_SCRATCH_BYTES


def build(force=True):
    """Compile every HIP source for gfx950 into libdynet_hip.so (hipcc cross-compiles without a GPU)."""
    args = ["make", "-C", CSRC_DIR, "-j8"]
    if force:
        args.append("-B")
    subprocess.run(args, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)


def declared_symbols():
    """Names of every entry point the public header declares."""
    with open(HEADER_PATH) as f:
        text = f.read()
    return sorted(set(re.findall(r"\b(dyhip_[a-z0-9_]+)\s*\(", text)))


# Argument types of every entry point as the header declares them (a test compares the two), so that the built library is all
# that an import needs: p an address, i int, u unsigned, f float, z size_t, q unsigned long long.
_ARGUMENTS = """
    accumulate:pzpp affine_forward:pzzzpppp argmax_cols:pzupp argmax_onehot_forward:pzuppp batch_reduce_workspace:zup
    clip_scale:pupfp clip_scale_norm:pupfpp cmult_backward:pzuupppuppz cmult_forward:pzuuppp const_minus_x_forward:pzfpp
    const_plus_x_forward:pzfpp constant:pzfp csum_backward:pzuupuppz csum_forward:pzuuppp cwise_backward:pipppppuppz
    cwise_backward_workspace:ppup cwise_forward:pippppp dense_to_sparse_assign:pippp dense_to_sparse_block_add:pipipp
    dense_to_sparse_subtract:pippp device_allocate:pizp device_count:p device_create:ipp device_destroy:p device_fork:pp
    device_ordinal:pp device_pool:pip device_scalar:pip device_set_gemm_handoff:pui device_set_sequence_blocks:pu
    device_set_stream_threshold:pz device_stream:pp device_sync:p device_wait:pp dropout_backward:pzppp
    dropout_forward:pzfppp gather_segments:puzpp gemm_nn:pzzzppfp gemm_nt:pzzzppfp gemm_nt_acc:pzzzppp
    gemm_strided_batched:piizzzpzpzfpzu gemm_tn:pzzzppfp gemm_tn_acc:pzzzppp gemm_uses_wide_tiles:piizzzp
    gemm_wide_segments:zzzuppp graph_begin_capture:p graph_destroy:p graph_end_capture:pp graph_launch:pp host_alloc:zp
    host_free:p last_error: layer_norm_backward:pzupppppppz layer_norm_backward_static:pzupppppp
    layer_norm_backward_workspace:zup layer_norm_forward:pzupppp log_softmax_backward:pzupppp log_softmax_forward:pzuppp
    logsumexp_cols:pzuppp logsumexp_dim_backward:pzzupppup logsumexp_dim_forward:pzzupupp
    logsumexp_node_backward:puzuppppuppz logsumexp_node_forward:puzuppp lookup_accumulate_grads:pupzupppz
    lookup_accumulate_grads_planned:pupzupppz lookup_accumulate_grads_planned_workspace:uzp
    lookup_accumulate_grads_workspace:uzup lookup_build_plan:pupupzpz lookup_forward:puppzupfp lookup_plan_bytes:up
    lookup_plan_invalid_ids:pupp lookup_plan_workspace:uup lstm_c_backward:puupppup lstm_c_forward:puuppp
    lstm_cell_backward:puupppppuppp lstm_cell_backward_packed:puupppppupppp lstm_cell_forward:puupppupippp
    lstm_cell_workspace:puupp lstm_gates_backward:puppuuppppupupppuppz lstm_gates_backward_workspace:uuuuip
    lstm_gates_dpre:puuppp lstm_gates_forward:puppuupppppupuippz lstm_gates_workspace:uuuuip lstm_h_backward:puupppup
    lstm_h_forward:puuppp lstm_pack_input:puupp lstm_pack_recurrent:pupp lstm_pack_recurrent_transposed:pupp
    lstm_pack_recurrent_transposed16:pupp lstm_pack_state:puupp lstm_pack_state16:puupp lstm_packed_state16_floats:uup
    lstm_packed_state_floats:uup lstm_recurrent_backward:puupppzp lstm_recurrent_backward_packed:puupppzp
    lstm_recurrent_forward:puupppzp lstm_sequence_backward:puuupppppppz lstm_sequence_forward:puuuppppippppz
    lstm_sequence_workspace:puuup lstm_step_backward_packed:puupppppppppp lstm_step_backward_packed_dropout:puuppppppppppp
    lstm_step_forward:puupppppippp lstm_step_forward_packed:puupppppipppp lstm_step_forward_packed_dropout:puuppppppipppp
    lstm_step_forward_x:puuuppppppippp lstm_step_supported:puup mean_elems_backward:pzupp mean_elems_forward:pzupp
    memcpy_d2d:pppz memcpy_d2h:pppz memcpy_h2d:pppz parallel_accumulate:piippp parallel_memcpy:piippp
    pick_range_backward:pzzzzzpp pick_range_forward:pzzzzzpp pnls_backward:pzupppp pnls_backward_assign:pzupppp
    pnls_forward:pzupppp pnls_forward_staged:pzuppp pool_allocate:pzp pool_capacity:pp pool_create_host:pzzp
    pool_destroy:p pool_free:p pool_num_blocks:pp pool_set_used:pz pool_used:pp pool_zero_allocated:p
    randomize_bernoulli:pzffp randomize_normal:pzffp randomize_uniform:pzffp reset_rng:pu rng_set_position:pq
    rng_state:pppp scale_copy:pzpfp sgd_update:pzppfff sgd_update_rows:pupzuppfpf sgd_update_scaled:pzppfpfi
    softmax_backward:pzuppppz softmax_forward:pzupppz softmax_rows_backward:pzzuppp softmax_rows_forward:pzzupp
    sparse_to_dense_assign:pippp sparse_to_dense_block_assign_and_multiply:pipifpp squared_l2norm:pzpppz
    squared_l2norm_rows:pupzupppz squared_l2norm_rows_workspace:up squared_l2norm_workspace:zp std_elems_backward:pzupppp
    std_elems_forward:pzupp sum_batches_backward:pzupp sum_batches_forward:pzupppz sum_forward:puzuppp timer_start:p
    timer_stop:pp unary_backward:pizppp unary_forward:piizpp zero:ppz
"""
_KINDS = {"p": C.c_void_p, "i": C.c_int, "u": C.c_uint, "f": C.c_float, "z": C.c_size_t, "q": C.c_ulonglong}


def _declare(dll):
    """With argument types calls may pass plain integers, floats and addresses: ctypes converts those faster than Python builds
    a ctypes object for each (a call of eight arguments 3.0 -> 2.0 us)."""
    for entry in _ARGUMENTS.split():
        name, kinds = entry.split(":")
        if hasattr(dll, "dyhip_" + name):
            getattr(dll, "dyhip_" + name).argtypes = [_KINDS[k] for k in kinds]


def _load():
    if not os.path.exists(LIB_PATH):
        build(force=False)
    if not os.path.exists(LIB_PATH):
        raise ImportError("libdynet_hip.so is missing and could not be built; there is no fallback path")
    return C.CDLL(LIB_PATH)


# ``cdll``: any ctypes objects as arguments; ``calls``: the same library for the package's own calls, with the argument types.
cdll = _load()
cdll.dyhip_last_error.restype = C.c_char_p
cdll.dyhip_last_error.argtypes = []
calls = _load()
_declare(calls)


def last_error():
    msg = cdll.dyhip_last_error()
    return msg.decode("utf-8", "replace") if msg else ""
