// Executor: kernel launches, whole-plan execution and host I/O (see k44_executor.hpp).
#include "k44_executor.hpp"

namespace k44_host {

// whole: whole-plan execution (folded / fused commands apply).
void K44GpuExecutorState::launch_aux(const AuxExec &a, bool whole) {
    __half *cv = canvas.p;
    switch (a.type) {
    case K44CmdType::RMSNORM_1D:
        if (whole && a.shift_with != SIZE_MAX) {
            const AuxExec &t = *aux[a.shift_with];
            const k44dev::RmsShift sh{cv + t.y_off, t.table.p,
                                      t.has_state ? cv + t.state_off : nullptr, t.rf, 0u,
                                      t.decode ? 0u : t.seq_len};
            const uint64_t *sl = a.norm_fold != SIZE_MAX ? fold_slots(a.norm_fold) : nullptr;
            const uint32_t n = a.norm_fold != SIZE_MAX ? norm_folds[a.norm_fold].tiles : 0u;
            K44_HIP(k44dev::launch_rmsnorm(cv + a.y_off, cv + a.src_off, a.table.p, a.D,
                                           a.stride, a.tokens, a.eps, stream, &sh, sl, n));
        } else if (whole && a.norm_fold != SIZE_MAX) {
            K44_HIP(k44dev::launch_rmsnorm(cv + a.y_off, cv + a.src_off, a.table.p, a.D,
                                           a.stride, a.tokens, a.eps, stream, nullptr,
                                           fold_slots(a.norm_fold), norm_folds[a.norm_fold].tiles));
        } else {
            K44_HIP(k44dev::launch_rmsnorm(cv + a.y_off, cv + a.src_off, a.table.p, a.D,
                                           a.stride, a.tokens, a.eps, stream));
        }
        break;
    case K44CmdType::SWIGLU_MUL_1D:
        if (whole && a.chain_inner != SIZE_MAX) {
            const AuxExec &in = *aux[a.chain_inner];
            K44_HIP(k44dev::launch_mul3(cv + a.y_off, cv + a.chain_other, cv + in.src_off,
                                        cv + in.src2_off, (uint64_t)a.D * a.stride, stream));
        } else {
            K44_HIP(k44dev::launch_mul(cv + a.y_off, cv + a.src_off, cv + a.src2_off,
                                       (uint64_t)a.D * a.stride, stream));
        }
        break;
    case K44CmdType::TOKEN_SHIFT_1D:
        K44_HIP(k44dev::launch_token_shift(cv + a.y_off, cv + a.src_off, a.table.p,
                                           a.has_state ? cv + a.state_off : nullptr, a.D,
                                           a.stride, a.tokens, a.rf, a.seq_len,
                                           a.decode ? 1 : 0, stream));
        break;
    case K44CmdType::EMBED_1D: {
        k44dev::EmbedCopy cp;
        if (whole && a.cp_fold != SIZE_MAX) {  // the first layer's compact token-shift state
            const NormFold &f = norm_folds[a.cp_fold];
            const AuxExec &T = *aux[f.shift];
            cp.src = cv + T.state_off;
            cp.sstride = 64u;
            cp.dst = shift_next.p + f.cur0;
            cp.dstride = 16u;
            cp.rows = T.D * (T.rf - 1u);
        }
        K44_HIP(k44dev::launch_embed(
            cv + a.y_off, a.table.p, ids.p, a.D, a.vocab, a.stride, a.tokens, stream,
            whole && a.slot_fold != SIZE_MAX
                ? reinterpret_cast<uint64_t *>(norm_slots.p) +
                      (norm_folds[a.slot_fold].slot0 + a.slot_tile0) * 32u
                : nullptr,
            cp));
        break;
    }
    case K44CmdType::S2D_2X2:
        K44_HIP(k44dev::launch_s2d(cv + a.y_off, cv + a.src_off, a.C, a.pin, a.pout, stream));
        K44_HIP(k44dev::launch_halo_clear(cv + a.y_off, a.out_channels, a.pout, stream));
        break;
    case K44CmdType::MAXPOOL_2X2:
        K44_HIP(k44dev::launch_maxpool2(cv + a.y_off, cv + a.src_off, a.C, a.pin, a.pout, stream));
        K44_HIP(k44dev::launch_halo_clear(cv + a.y_off, a.out_channels, a.pout, stream));
        break;
    case K44CmdType::MAXPOOL_5X5:
        K44_HIP(k44dev::launch_maxpool5(cv + a.y_off, cv + a.src_off, a.C, a.pin, a.pout, stream));
        K44_HIP(k44dev::launch_halo_clear(cv + a.y_off, a.out_channels, a.pout, stream));
        break;
    case K44CmdType::UPSAMPLE_2X:
        K44_HIP(k44dev::launch_upsample2(cv + a.y_off, cv + a.src_off, a.C, a.pin, a.pout, stream));
        K44_HIP(k44dev::launch_halo_clear(cv + a.y_off, a.out_channels, a.pout, stream));
        break;
    case K44CmdType::SCATTER_UP2X2:
        K44_HIP(k44dev::launch_scatter_up2(cv + a.y_off, cv + a.src_off, a.C, a.D, a.pin,
                                           a.pout, stream));
        K44_HIP(k44dev::launch_halo_clear(cv + a.y_off, a.out_channels, a.pout, stream));
        break;
    case K44CmdType::ARGMAX_1D:
        K44_HIP(k44dev::launch_argmax(ids.p, hist_steps ? history.p : nullptr, step_ctr.p,
                                      hist_steps, cv + a.src_off, a.D, a.stride, a.tokens,
                                      scratch.p, stream));
        break;
    default:
        throw std::runtime_error("unsupported aux command");
    }
}

void K44GpuExecutorState::launch_mfma_group(const k44dev::MfmaGroup &d, uint32_t nt, uint32_t mt, uint32_t rows,
                       uint32_t items, uint32_t epi_items, bool dma, const k44dev::DmaShape &ds,
                       uint32_t prod, uint32_t max_items, bool mis,
                       const k44dev::NarrowPre &pre) {
    if (mt == 16u)  // narrow (<= 16 tokens)
        K44_HIP(k44dev::launch_mfma_narrow(d, nt, items, stream, prod, max_items, pre));
    else if (dma)
        K44_HIP(k44dev::launch_mfma_dma(d, nt, items, stream, ds));
    else
        K44_HIP(k44dev::launch_mfma_tile(d, nt, mt, rows, items, stream, mis));
    if (epi_items) K44_HIP(k44dev::launch_splitk_epilogue(d, epi_items, stream));
}

void K44GpuExecutorState::launch_jobs(const WaveExec &w) {
    k44dev::JobArgs a{};
    a.X = canvas.p + w.rk_base;
    a.roff = w.roff.p;
    a.Wf = w.w.p;
    a.jmap = w.jmap.p;
    a.koff = w.koff.p;
    a.part = scratch.p;
    a.ksteps = w.jb_ksteps;
    a.tiles = w.jb_tiles;
    a.ttiles = w.tokens / 64u;
    a.tokens = w.tokens;
    a.S = w.S;
    K44_HIP(k44dev::launch_mfma_jobs(a, stream));
    k44dev::JobReduceArgs r{};
    r.part = scratch.p;
    r.bias = w.bias.p;
    r.cmap = w.cmap.p;
    r.Y = canvas.p + w.y_off;
    r.R = w.has_res ? canvas.p + w.res_off : nullptr;
    r.out_stride = w.out_stride;
    r.cout = w.cout;
    r.K = w.K;
    r.tokens = w.tokens;
    r.act = w.act;
    K44_HIP(k44dev::launch_jobs_reduce(r, stream));
}

void K44GpuExecutorState::launch_list(const WaveExec &w) {
    k44dev::RowListArgs a{};
    a.X = canvas.p + w.rk_base;
    a.roff = w.roff.p;
    a.W = w.w.p;
    a.bias = w.bias.p;
    a.cmap = w.cmap.p;
    a.Y = canvas.p + w.y_off;
    a.R = w.has_res ? canvas.p + w.res_off : nullptr;
    a.out_stride = w.out_stride;
    a.cout = w.cout;
    a.cluster = w.cluster;
    a.B = w.K * w.S;
    a.steps = (a.B + 31u) / 32u;
    a.ttiles = w.tokens / 64u;
    a.act = w.act;
    K44_HIP(k44dev::launch_row_list(a, w.rl_kw, stream));
}

k44dev::RowsArgs K44GpuExecutorState::rows_args(const WaveExec &w, bool fused) const {
    k44dev::RowsArgs a{};
    a.X = canvas.p + w.rk_base;
    a.roff = w.roff.p;
    a.Wf = w.w.p;
    a.bias = w.bias.p;
    a.cmap = w.cmap.p;
    a.Y = canvas.p + (fused ? w.y_off_run : w.y_off);
    a.R = w.has_res ? canvas.p + w.res_off : nullptr;
    a.tile_x = w.tile_x.p;
    a.tile_y = w.tile_y.p;
    a.out_stride = w.out_stride;
    a.B = w.rk_B;
    a.ksteps = w.rk_ksteps;
    a.blocks = w.cluster / 16u;
    a.subs = w.rk_subs;
    a.ttiles = w.rk_ttiles();
    a.act = w.act;
    a.vec = w.rk_vec;
    if (w.tile2d && w.masked) {
        a.mask_w = w.plane.W;
        a.mask_h = w.plane.H;
        a.mask_wpad = w.plane.W_pad;
        a.mask_tpf = w.tiles_per_frame;
    }
    return a;
}

// One wave alone, as compiled (a wave's output never moves past the canvas unless folded).
void K44GpuExecutorState::launch_rows(const WaveExec &w) {
    k44dev::RowsLaunch l;
    l.one = rows_args(w, false);
    if (w.tile2d && !w.plane.tok64 && w.rk_mis) {
        l.halo = canvas.p + w.y_off;
        l.halo_planes = w.cout * w.plane.frames;
        l.plane = w.plane;
    }
    K44_HIP(k44dev::launch_mfma_rows(l, w.rows * w.rk_subs, w.rk_ttiles(), w.rk_nb, w.rk_kw,
                                     w.rk_mis, stream));
}

void K44GpuExecutorState::launch_mfma(const WaveExec &w) {
    const k44dev::MfmaGroup d{w.one_args.p, w.one_start.p, 1u, xcd_order};
    launch_mfma_group(d, w.cluster, w.mt, w.rows_per_stage, w.items, w.epi_items, w.dma,
                      w.dshape, 0u, w.items, w.mis, w.one_pre);
}

void K44GpuExecutorState::launch_group(const MfmaGroupExec &g) {
    if (g.rowsk) {
        const WaveExec &w = *waves[g.members[0]];
        k44dev::RowsLaunch l;
        if (g.members.size() > 1u) {
            l.waves = g.rk_args.p;
            l.start = g.start.p;
            l.n = (uint32_t)g.members.size();
        } else {
            l.one = rows_args(w, true);
        }
        K44_HIP(k44dev::launch_mfma_rows(l, g.rk_cols, g.rk_ttiles, w.rk_nb, w.rk_kw, w.rk_mis,
                                         stream));
        return;
    }
    const k44dev::MfmaGroup d{g.args.p, g.start.p, (uint32_t)g.members.size(), xcd_order};
    launch_mfma_group(d, g.nt, g.mt, g.rows, g.items, g.epi_items, g.dma, g.dshape,
                      g.prod, g.max_items, g.mis, g.pre);
}

void K44GpuExecutorState::launch_wave(const WaveExec &w) {
    if (w.jb_tiles) {
        launch_jobs(w);
        return;
    }
    if (w.rl_kw) {
        launch_list(w);
        return;
    }
    if (w.rowsk) {
        launch_rows(w);
        if (w.tile2d && (w.plane.tok64 || !w.rk_mis))
            K44_HIP(k44dev::launch_halo_clear(canvas.p + w.y_off, w.cout, w.plane, stream));
        return;
    }
    if (w.mfma) {
        launch_mfma(w);
        if (w.tile2d)
            K44_HIP(k44dev::launch_halo_clear(canvas.p + w.y_off, w.cout, w.plane, stream));
        return;
    }
    if (w.tile2d) {
        k44dev::GatherTileArgs a{};
        a.X = canvas.p;
        a.seg = w.seg.p;
        a.W = w.w.p;
        a.bias = w.bias.p;
        a.cmap = w.cmap.p;
        a.Y = canvas.p + w.y_off;
        a.R = w.has_res ? canvas.p + w.res_off : nullptr;
        a.tile_x = w.tile_x.p;
        a.tile_y = w.tile_y.p;
        a.step = w.step;
        a.K = w.K;
        a.S = w.S;
        a.cluster = w.cluster;
        a.cout = w.cout;
        a.tiles = w.tiles;
        a.out_stride = w.plane.channel_stride;
        a.act = w.act;
        a.plane = w.plane;
        a.tiles_per_frame = w.tiles_per_frame;
        a.masked = w.masked;
        K44_HIP(k44dev::launch_gather_tile(a, stream));
        K44_HIP(k44dev::launch_halo_clear(canvas.p + w.y_off, w.cout, w.plane, stream));
        return;
    }
    k44dev::GatherDotArgs a{};
    a.X = canvas.p;
    a.seg = w.seg.p;
    a.W = w.w.p;
    a.bias = w.bias.p;
    a.cmap = w.cmap.p;
    a.Y = canvas.p + w.y_off;
    a.R = w.has_res ? canvas.p + w.res_off : nullptr;
    a.step = w.step;
    a.K = w.K;
    a.S = w.S;
    a.n_batch = w.n_batch;
    a.cluster = w.cluster;
    a.cout = w.cout;
    a.out_stride = w.out_stride;
    a.act = w.act;
    if (w.stream_kernel)
        K44_HIP(k44dev::launch_gather_stream(a, w.tokens, stream, w.stream_loads));
    else
        K44_HIP(k44dev::launch_gather_dot(a, w.slab, w.ksplit, w.tokens, stream, w.lane8,
                                          w.stream_loads, w.weights_in_lds, w.misaligned));
}

void K44GpuExecutorState::launch_op(size_t i) {
    const auto &op = ops.at(i);
    if (op.first)
        launch_wave(*waves[op.second]);
    else
        launch_aux(*aux[op.second]);
}

void K44GpuExecutorState::launch_ops(size_t first, size_t n) {
    const size_t end = n == SIZE_MAX ? runs.size() : std::min(runs.size(), first + n);
    for (size_t i = first; i < end; ++i) {
        const auto &r = runs[i];
        if (r.first == 0)
            launch_aux(*aux[r.second], true);
        else if (r.first == 1)
            launch_wave(*waves[r.second]);
        else
            launch_group(*groups[r.second]);
    }
}

// One plan run on the executor stream: kernel by kernel, or as one replay of a HIP graph
// captured from the same launches (no memset/memcpy nodes in it).
void K44GpuExecutorState::execute_plan() {
    if (prog_active) {  // one launch: nothing to capture
        K44_HIP(k44dev::launch_program(prog_args, prog_grid, stream));
        return;
    }
    if (!use_graph) {
        launch_ops();
        return;
    }
    if (!graph_exec) {
        K44_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        try {
            launch_ops();
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(stream, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        K44_HIP(hipStreamEndCapture(stream, &graph));
        K44_HIP(hipGraphInstantiate(&graph_exec, graph, nullptr, nullptr, 0));
    }
    K44_HIP(hipGraphLaunch(graph_exec, stream));
}

void K44GpuExecutorState::set_history(uint32_t steps) {
    if (!id_tokens) throw std::runtime_error("plan has no token-id buffer (no embed/argmax)");
    K44_HIP(hipStreamSynchronize(stream));
    drop_graph();  // the history pointer is baked into captured launches
    history.alloc((size_t)std::max(1u, steps) * id_tokens);
    hist_steps = steps;
    K44_HIP(hipMemsetAsync(history.p, 0, history.n * 4u, stream));
    K44_HIP(hipMemsetAsync(step_ctr.p, 0, 4u, stream));
    K44_HIP(hipStreamSynchronize(stream));
    if (prog_active) build_program();  // the history pointer is in its argmax stage
}

static k44dev::FrameLayout frame_layout(const K44ResDesc &L, uint32_t H, uint32_t W) {
    k44dev::FrameLayout f{};
    f.channel_stride = L.channel_stride;
    f.H = H;
    f.W = W;
    f.x_step = 1u;
    if (!L.is_1d_tokens) {
        f.y0 = 1u;
        f.x0 = L.is_image_token64 ? 1u : 4u;
        f.x_step = L.is_image_token64 ? 64u : 1u;
        f.row_stride = L.W_pad * f.x_step;
    }
    return f;
}

// Input channels cross to the device as they are and are converted there: small inputs from the
// page-locked ring, which the kernel reads in place (a copy of its own would cost more than the
// transfer: a block over 640 x 3 values 79 -> 53 us per call), larger ones at most kInStage bytes
// or one channel at a time, in stream order.  Whole channels are written: the region may hold
// another tensor's data from the last run.
void K44GpuExecutorState::upload_input_f32(const float *in, size_t n) {
    constexpr size_t kInStage = 16u << 20, kInPlace = 256u << 10;
    const k44dev::FrameLayout f = frame_layout(layout(plan_meta.input_res_key),
                                                plan_meta.input_h, plan_meta.input_w);
    const size_t per = (size_t)f.H * f.W;
    const uint32_t C = plan_meta.input_c;
    n = std::min(n, per * C);
    uint16_t *region = reinterpret_cast<uint16_t *>(canvas.p + plan_meta.input_off);
    if (n * 4u <= kInPlace) {
        std::memcpy(ring.p, in, n * 4u);
        K44_HIP(k44dev::launch_import_f32(region, reinterpret_cast<const float *>(ring.p), n, C, f,
                                          stream));
        return;
    }
    const uint32_t step = (uint32_t)std::min<size_t>(C, std::max<size_t>(1u, kInStage / (per * 4u)));
    if (in_stage.n < per * step) in_stage.alloc(per * step);
    for (uint32_t c = 0; c < C; c += step) {
        const uint32_t nc = std::min(step, C - c);
        const size_t first = per * c;
        const size_t cnt = first < n ? std::min(n - first, per * nc) : 0u;
        if (cnt)
            K44_HIP(hipMemcpyAsync(in_stage.p, in + first, cnt * 4u, hipMemcpyHostToDevice, stream));
        K44_HIP(k44dev::launch_import_f32(region + (size_t)c * f.channel_stride, in_stage.p, cnt,
                                          nc, f, stream));
    }
}

// How a read reaches [p, p + bytes): in place at `direct` if all of it is one page-locked host
// allocation or memory of the executor's GPU, aligned as the kernels store; else through the ring,
// by the runtime's copy to memory of another GPU (`device`), by the host to its own.
struct Target {
    void *direct;
    bool device;
};
static Target target_of(void *p, size_t bytes, size_t align) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return {nullptr, false};
    }
    const bool device = at.type == hipMemoryTypeDevice;
    int gpu = at.device;
    if (device) K44_HIP(hipGetDevice(&gpu));
    if ((!device && at.type != hipMemoryTypeHost) || at.device != gpu ||
        !at.devicePointer || reinterpret_cast<uintptr_t>(at.devicePointer) % align != 0u)
        return {nullptr, device};
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, reinterpret_cast<hipDeviceptr_t>(at.devicePointer)) !=
        hipSuccess) {
        (void)hipGetLastError();
        return {nullptr, device};
    }
    const size_t skip = static_cast<char *>(at.devicePointer) - static_cast<char *>(base);
    return {skip <= size && bytes <= size - skip ? at.devicePointer : nullptr, device};
}

// Fills caller memory from a kernel and waits for it: fill(target, first byte, bytes) enqueues a
// kernel that writes that part of the output to `target`, `align` bytes a value.  Page-locked
// destinations are written in place, without a staging buffer and the copy after it (0.5 MB of a
// 64-token wave: 43 -> 33 us around the plan's run); others through the ring, one chunk copied out
// while a kernel writes the next (a copy to pageable memory of 4 MB takes 250 us, the ring 187; of
// 1 GB 64 ms, 44).
template <typename Fill>
void K44GpuExecutorState::to_host(void *dst, size_t bytes, size_t align, Fill &&fill) {
    const Target to = target_of(dst, bytes, align);
    if (to.direct) {
        fill(to.direct, 0u, bytes);
        K44_HIP(hipStreamSynchronize(stream));
        return;
    }
    std::lock_guard<std::recursive_mutex> lk(io);
    constexpr size_t kChunk = HostRing::kChunk;
    auto out = [&](size_t at, const char *from, size_t n) {
        char *d = static_cast<char *>(dst) + at;
        if (to.device)
            K44_HIP(hipMemcpy(d, from, n, hipMemcpyDefault));
        else
            std::memcpy(d, from, n);
    };
    if (bytes <= kChunk) {
        fill(ring.p, 0u, bytes);
        K44_HIP(hipStreamSynchronize(stream));
        out(0u, ring.p, bytes);
        return;
    }
    const size_t chunks = (bytes + kChunk - 1u) / kChunk;
    auto take = [&](size_t i) {
        K44_HIP(hipEventSynchronize(ring.ev[i & 1u]));
        out(i * kChunk, ring.p + (i & 1u) * kChunk, std::min(kChunk, bytes - i * kChunk));
    };
    for (size_t i = 0; i < chunks; ++i) {
        if (i >= 2u) take(i - 2u);
        fill(ring.p + (i & 1u) * kChunk, i * kChunk, std::min(kChunk, bytes - i * kChunk));
        K44_HIP(hipEventRecord(ring.ev[i & 1u], stream));
    }
    take(chunks - 2u);
    take(chunks - 1u);
}

void K44GpuExecutorState::download_output_f32(float *out, size_t n) {
    const k44dev::FrameLayout f = frame_layout(layout(plan_meta.output_res_key),
                                                plan_meta.output_h, plan_meta.output_w);
    const uint16_t *region = reinterpret_cast<const uint16_t *>(canvas.p + plan_meta.output_off);
    to_host(out, n * 4u, 4u, [&](void *to, size_t first, size_t bytes) {
        K44_HIP(k44dev::launch_export_f32(static_cast<float *>(to), region, first / 4u, bytes / 4u,
                                          f, stream));
    });
}

void K44GpuExecutorState::read_rows(uint16_t *dst, uint64_t off, uint64_t rows, uint64_t row_stride,
                                    uint64_t cols) {
    const uint16_t *src = reinterpret_cast<const uint16_t *>(canvas.p + off);
    to_host(dst, rows * cols * 2u, 2u, [&](void *to, size_t first, size_t bytes) {
        K44_HIP(k44dev::launch_pack_rows(static_cast<uint16_t *>(to), src, first / 2u, bytes / 2u,
                                         row_stride, cols, stream));
    });
}

int K44GpuExecutorState::infer_f32(const float *in, int in_elems, float *out, int out_elems, float *ms_out) {
    if (!initialized) throw std::runtime_error("executor not initialised");
    std::lock_guard<std::recursive_mutex> lk(io);  // (the ring holds a small input until it ran)
    upload_input_f32(in, (size_t)std::max(0, in_elems));
    K44_HIP(hipEventRecord(ev0, stream));
    execute_plan();
    K44_HIP(hipEventRecord(ev1, stream));
    download_output_f32(out, std::min((size_t)std::max(0, out_elems),
                                      (size_t)plan_meta.output_c * plan_meta.output_h *
                                          plan_meta.output_w));
    K44_HIP(hipEventSynchronize(ev1));
    float ms = 0.0f;
    K44_HIP(hipEventElapsedTime(&ms, ev0, ev1));
    if (ms_out) *ms_out = ms;
    return 0;
}

}  // namespace k44_host
