// The operator's and the layer's training step as native autograd functions (included by gdn_host.cpp): forward and backward allocate,
// launch and return without the interpreter.  Small steps were bound by it: 110 - 160 us of host time for the operator's step, 1390 us
// for the layer's (some ninety launches, each through an autograd node of its own), whatever the size of the tensors.
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

template <typename T = void>
T* ptr_of(const at::Tensor& t) { return t.defined() ? (T*)t.data_ptr() : nullptr; }
at::Tensor to_f32(const at::Tensor& t) { return t.defined() ? t.detach().to(at::kFloat).contiguous() : t; }
at::Tensor sum_rows(const at::Tensor& part, at::ScalarType type, at::IntArrayRef shape, void* stream) {       // over the first dimension
    at::Tensor out = empty_on(part.device(), type, shape);
    check_rc(p_sum_rows((const float*)part.data_ptr(), out.data_ptr(), part.size(0), out.numel(), code_of(type), stream), "gdn_sum_rows");
    return out;
}

// A saved tensor as the kernels read it.  Saved-tensor hooks (offloading, checkpointing, compression) may hand back another layout,
// place or type than they were given.
at::Tensor saved(const at::Tensor& t, at::ScalarType type, c10::Device dev) {
    if (!t.defined() || (t.scalar_type() == type && t.device() == dev && t.is_contiguous() && aligned16(t.data_ptr()))) return t;
    const at::Tensor r = t.to(at::TensorOptions().dtype(type).device(dev)).contiguous();
    return aligned16(r.data_ptr()) ? r : r.clone();
}

// What a call of the operator is made of besides its tensors.
struct ChunkCall {
    int64_t B, T, H, HV, K, V, N, num_chunks;
    double scale;
    uint32_t flags;                    // as gdn_chunk_fwd takes them
    bool out_final, vfirst;
    bool whole = true;                 // the boundaries cover every token
};

void chunk_forward(const ChunkCall& c, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const void* g, const void* beta, int gb,
                   const at::Tensor& A_log, const at::Tensor& dt_bias, const at::Tensor& h0, const at::Tensor& cu, const at::Tensor& table,
                   const at::Tensor& offsets, at::Tensor& o, at::Tensor& ht) {
    const c10::Device dev = q.device();
    const size_t ws_bytes = p_chunk_workspace_bytes(c.N, c.T, c.num_chunks, c.H, c.HV, c.K, c.V, cu.defined() ? 1 : 0, c.flags);
    TORCH_CHECK(ws_bytes > 0, "gdn_chunk_fwd does not cover K=", c.K, ", V=", c.V);
    o = empty_on(dev, v.scalar_type(), {c.B, c.T, c.HV, c.V});
    if (c.out_final) ht = c.vfirst ? empty_on(dev, at::kFloat, {c.N, c.HV, c.V, c.K}) : empty_on(dev, at::kFloat, {c.N, c.HV, c.K, c.V});
    const at::Tensor ws = empty_on(dev, at::kByte, {(int64_t)ws_bytes});
    check_rc(p_chunk_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), g, beta, ptr_of<float>(A_log), ptr_of<float>(dt_bias), ptr_of<float>(h0), ptr_of<float>(ht),
                         o.data_ptr(), ptr_of(cu), ptr_of(table), ptr_of(offsets), ws.data_ptr(), ws_bytes, c.B, c.T, c.H, c.HV, c.K, c.V, c.N,
                         c.num_chunks, (float)c.scale, code_of(q.scalar_type()), gb, c.flags, stream_of(dev)), "gdn_chunk_fwd");
}

// dg, db: gradients of the gate and of beta (behind their activations), fp32 [B,T,HV]
struct ChunkGrads { at::Tensor dq, dk, dv, dg, db, dh0; };
ChunkGrads chunk_backward(const ChunkCall& c, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const void* g, const void* beta, int gb,
                          const at::Tensor& A_log, const at::Tensor& dt_bias, const at::Tensor& h0, const at::Tensor& cu, const at::Tensor& table,
                          const at::Tensor& offsets, const at::Tensor& dout, const at::Tensor& dht) {
    const c10::Device dev = q.device();
    const at::ScalarType type = q.scalar_type();
    const uint32_t flags = c.flags & (GDN_FLAG_QK_L2NORM | GDN_FLAG_BETA_SIGMOID | GDN_FLAG_NEG_EIGVAL | GDN_FLAG_CU_INT32 | GDN_FLAG_SEQ_ORDER);
    // (tokens of a packed tensor outside every sequence get zero gradients)
    auto alloc = [&](at::ScalarType s, at::IntArrayRef shape) { return c.whole ? empty_on(dev, s, shape) : at::zeros(shape, at::TensorOptions().dtype(s).device(dev)); };
    ChunkGrads r;
    r.dq = alloc(type, {c.B, c.T, c.H, c.K}); r.dk = alloc(type, {c.B, c.T, c.H, c.K}); r.dv = alloc(type, {c.B, c.T, c.HV, c.V});
    r.dg = alloc(at::kFloat, {c.B, c.T, c.HV}); r.db = alloc(at::kFloat, {c.B, c.T, c.HV});
    at::Tensor h = h0, d = dht;
    if (c.vfirst && h.defined()) h = h.transpose(-1, -2).contiguous();
    if (d.defined()) d = (c.vfirst ? d.transpose(-1, -2) : d).to(at::kFloat).contiguous();
    if (h0.defined()) r.dh0 = empty_on(dev, at::kFloat, {c.N, c.HV, c.K, c.V});
    const size_t ws_bytes = p_chunk_bwd_heads_workspace_bytes(c.num_chunks, c.H, c.HV, c.K, c.V, c.B * c.T, flags);
    const at::Tensor ws = empty_on(dev, at::kByte, {(int64_t)std::max<size_t>(ws_bytes, 1)});
    check_rc(p_chunk_bwd_heads(q.data_ptr(), k.data_ptr(), v.data_ptr(), g, beta, ptr_of<float>(A_log), ptr_of<float>(dt_bias), ptr_of<float>(h),
                               dout.data_ptr(), ptr_of<float>(d), r.dq.data_ptr(), r.dk.data_ptr(), r.dv.data_ptr(), (float*)r.dg.data_ptr(),
                               (float*)r.db.data_ptr(), ptr_of<float>(r.dh0), ptr_of(cu), ptr_of(table), ptr_of(offsets), ws.data_ptr(), ws_bytes,
                               c.B, c.T, c.H, c.HV, c.K, c.V, c.N, c.num_chunks, (float)c.scale, code_of(type), gb, flags, stream_of(dev)), "gdn_chunk_bwd_heads");
    if (c.vfirst && r.dh0.defined()) r.dh0 = r.dh0.transpose(-1, -2).contiguous();
    return r;
}

int64_t gate_parts(int64_t rows, int64_t HV) { return std::max<int64_t>(1, std::min<int64_t>(256, rows * HV / 256)); }

// ---- the operator ----
struct ChunkTrain : torch::autograd::Function<ChunkTrain> {
    typedef std::optional<at::Tensor> Maybe;
    static variable_list forward(AutogradContext* ctx, const Variable& q, const Variable& k, const Variable& v, const Maybe& g_, const Variable& beta,
                                 const Maybe& h0_, const Maybe& A_log_, const Maybe& dt_bias_, const Maybe& cu_, const Maybe& table_,
                                 const Maybe& offsets_, const ChunkCall& c) {
        const at::Tensor g = g_.value_or(at::Tensor()), h0 = h0_.value_or(at::Tensor()), A_log = A_log_.value_or(at::Tensor()), dt_bias = dt_bias_.value_or(at::Tensor()),
                         cu = cu_.value_or(at::Tensor()), table = table_.value_or(at::Tensor()), offsets = offsets_.value_or(at::Tensor());
        const at::Tensor A = to_f32(A_log), dt = to_f32(dt_bias);
        at::Tensor o, ht;
        chunk_forward(c, q, k, v, ptr_of(g), beta.data_ptr(), gb_code(g, beta), A, dt, h0, cu, table, offsets, o, ht);
        ctx->save_for_backward({q, k, v, g, beta, h0, A_log, dt_bias, cu, table, offsets});
        ctx->saved_data["dims"] = std::vector<int64_t>{c.B, c.T, c.H, c.HV, c.K, c.V, c.N, c.num_chunks, (int64_t)c.flags, c.out_final, c.vfirst, c.whole};
        ctx->saved_data["scale"] = c.scale;
        ctx->saved_data["types"] = std::vector<int64_t>{(int64_t)q.scalar_type(), (int64_t)(g.defined() ? g : beta).scalar_type(), (int64_t)beta.scalar_type()};
        ctx->saved_data["device"] = q.device();
        ctx->set_materialize_grads(false);
        if (!c.out_final) return {o};
        return {o, ht};
    }
    static int gb_code(const at::Tensor& g, const at::Tensor& beta) {
        const int cb = code_of(beta.scalar_type()), cg = g.defined() ? code_of(g.scalar_type()) : cb;
        return cb == cg ? cg : GDN_GB_DTYPES(cg, cb);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const c10::Device dev = ctx->saved_data["device"].toDevice();
        const c10::DeviceGuard guard(dev);
        const std::vector<int64_t> types = ctx->saved_data["types"].toIntVector();
        auto s = ctx->get_saved_variables();
        for (int i = 0; i < 5; ++i) s[i] = saved(s[i], (at::ScalarType)types[std::max(0, i - 2)], dev);
        for (int i = 5; i < (int)s.size(); ++i)
            if (s[i].defined()) s[i] = saved(s[i], i == 5 ? at::kFloat : s[i].scalar_type(), dev);
        const at::Tensor &q = s[0], &k = s[1], &v = s[2], &g = s[3], &beta = s[4], &h0 = s[5], &A_log = s[6], &dt_bias = s[7];
        const std::vector<int64_t> n = ctx->saved_data["dims"].toIntVector();
        const ChunkCall c{n[0], n[1], n[2], n[3], n[4], n[5], n[6], n[7], ctx->saved_data["scale"].toDouble(), (uint32_t)n[8], n[9] != 0, n[10] != 0, n[11] != 0};
        void* stream = stream_of(dev);
        at::Tensor dout = grads[0].defined() ? grads[0].to(v.scalar_type()).contiguous() : at::zeros_like(v);
        if (!aligned16(dout.data_ptr())) dout = dout.clone();
        const at::Tensor A = to_f32(A_log), dt = to_f32(dt_bias);
        const at::Tensor dht = grads.size() > 1 ? grads[1] : at::Tensor();
        ChunkGrads r = chunk_backward(c, q, k, v, ptr_of(g), beta.data_ptr(), gb_code(g, beta), A, dt, h0, s[8], s[9], s[10], dout, dht);
        at::Tensor dA, ddt, dg = r.dg, db = r.db;
        const bool bsig = c.flags & GDN_FLAG_BETA_SIGMOID;
        if (A.defined() || bsig) {
            const int64_t rows = c.B * c.T, parts = gate_parts(rows, c.HV);
            const bool gate = A.defined();
            dg = gate ? at::empty_like(g) : r.dg;
            db = at::empty_like(beta);
            const at::Tensor part = gate ? empty_on(q.device(), at::kFloat, {parts, 2, c.HV}) : at::Tensor();
            check_rc(p_gate_bwd(gate ? (const float*)r.dg.data_ptr() : nullptr, (const float*)r.db.data_ptr(), gate ? g.data_ptr() : nullptr, beta.data_ptr(),
                                ptr_of<float>(A), ptr_of<float>(dt), gate ? dg.data_ptr() : nullptr, db.data_ptr(), ptr_of<float>(part), rows, c.HV, parts,
                                c.HV, c.HV, c.HV, c.HV, 0, 0, gate ? code_of(g.scalar_type()) : GDN_DTYPE_F32, code_of(beta.scalar_type()),
                                bsig ? (c.flags & GDN_FLAG_NEG_EIGVAL ? 2.f : 1.f) : 0.f, stream), "gdn_gate_bwd");
            if (gate) {
                const at::Tensor sums = sum_rows(part, at::kFloat, {2, c.HV}, stream);
                dA = sums[0].to(A_log.scalar_type()).view(A_log.sizes());
                if (dt.defined()) ddt = sums[1].to(dt_bias.scalar_type()).view(dt_bias.sizes());
            }
        }
        if (!g.defined()) dg = at::Tensor();
        else if (dg.scalar_type() != g.scalar_type()) dg = dg.to(g.scalar_type());
        if (db.scalar_type() != beta.scalar_type()) db = db.to(beta.scalar_type());
        return {r.dq, r.dk, r.dv, dg, db, r.dh0, dA, ddt, Variable(), Variable(), Variable(), Variable()};
    }
};

// (q, k, v, g, beta, scale, initial_state, output_final_state, state_v_first, cu_seqlens, chunk_indices, scan_tables, A_log, dt_bias,
//  flags, whole); as chunk_fwd, for calls that need gradients.  None: not a call for the native path
PyObject* chunk_train(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 16) { PyErr_SetString(PyExc_TypeError, "gdn_host.chunk_train takes 16 arguments"); return nullptr; }
    ChunkArgs x;
    if (!chunk_args(a, x)) { if (PyErr_Occurred()) return nullptr; Py_RETURN_NONE; }
    const Dims& d = x.d;
    if (!((d.K == 64 && d.V == 64) || (d.K == 128 && d.V == 128) || (d.K == 256 && d.V % 128 == 0))) Py_RETURN_NONE;
    const ChunkCall c{d.B, d.T, d.H, d.HV, d.K, d.V, x.N, x.num_chunks, x.scale, x.flags, truth(a[7]), truth(a[8]), truth(a[15])};
    auto var = [](const Arg& t) { return t ? ChunkTrain::Maybe(*t.t) : ChunkTrain::Maybe(); };
    variable_list r;
    {
        const NoGil free;
        r = ChunkTrain::apply(*x.q.t, *x.k.t, *x.v.t, var(x.g), *x.beta.t, var(x.h0), var(x.A_log), var(x.dt_bias), var(x.cu), var(x.table), var(x.offsets), c);
    }
    return pair(r[0], r.size() > 1 ? r[1] : at::Tensor());
    END_HANDLE_TH_ERRORS
}

// ---- the layer ----
// tiles of 64 tokens per workgroup of the convolution's backward (modules/convolution.py: conv_bwd_run)
int64_t conv_bwd_run(int64_t num_tiles, int64_t D) {
    int64_t run = 8;
    while (run > 1 && (D + 255) / 256 * ((num_tiles + run - 1) / run) < 1024) run /= 2;
    return run;
}

// Projections of q, k, v, the gate and beta in one product with one matrix (and one product each for its two gradients: the six of a
// layer on their own left the small ones at 2 % of the matrix cores and added up five gradients of x), convolutions read and write
// slices of it; then the operator, the gated norm, the output projection.
struct LayerTrain : torch::autograd::Function<LayerTrain> {
    enum { X, QW, KW, VW, AW, BW, GW, OW, QC, KC, VC, A_LOG, DT, NW, INPUTS };
    static variable_list forward(AutogradContext* ctx, at::TensorList in, int64_t heads, bool neg, double eps) {
        const at::Tensor& x = in[X];
        const c10::Device dev = x.device();
        const at::ScalarType type = x.scalar_type();
        void* stream = stream_of(dev);
        const int code = code_of(type);
        const int64_t B = x.size(0), T = x.size(1), hidden = x.size(2), rows = B * T, kd = in[QW].size(0), vd = in[VW].size(0), HV = in[AW].size(0);
        const int64_t K = kd / heads, V = vd / HV, W = in[QC].size(-1), used = 2 * kd + vd + 2 * HV, ld = (used + 15) / 16 * 16;
        at::Tensor w = empty_on(dev, type, {ld, hidden});
        {
            std::vector<at::Tensor> parts{in[QW], in[KW], in[VW], in[AW], in[BW]};
            if (ld > used) parts.push_back(at::zeros({ld - used, hidden}, w.options()));
            at::cat_out(w, parts, 0);
        }
        const at::Tensor x2 = x.reshape({rows, hidden});
        const at::Tensor p = at::mm(x2, w.t());                                     // [rows][q | k | v | gate | beta | padding]
        const at::Tensor gate = at::mm(x2, in[GW].t());
        at::Tensor qkv[3];
        int64_t at = 0;
        for (int i = 0; i < 3; ++i) {
            const int64_t D = i < 2 ? kd : vd;
            qkv[i] = empty_on(dev, type, {B, T, i < 2 ? heads : HV, i < 2 ? K : V});
            check_rc(p_conv_fwd((const char*)p.data_ptr() + at * 2, in[QC + i].data_ptr(), nullptr, nullptr, nullptr, qkv[i].data_ptr(), nullptr, nullptr,
                                B, T, D, W, B, T * ld, ld, code, code, GDN_DTYPE_F32, GDN_ACT_SILU, 0, stream), "gdn_causal_conv1d_fwd");
            at += D;
        }
        const at::Tensor gb = p.narrow(1, at, 2 * HV).contiguous();                 // [rows][gate | beta]
        const at::Tensor graw = gb.narrow(1, 0, HV).contiguous(), braw = gb.narrow(1, HV, HV).contiguous();
        const at::Tensor A = to_f32(in[A_LOG]), dt = to_f32(in[DT]);
        const ChunkCall c = call_of(B, T, heads, HV, K, V, neg);
        at::Tensor o, none;
        chunk_forward(c, qkv[0], qkv[1], qkv[2], graw.data_ptr(), braw.data_ptr(), code, A, dt, none, none, none, none, o, none);
        const at::Tensor y = empty_on(dev, type, {rows, vd}), rstd = empty_on(dev, at::kFloat, {rows * HV});
        check_rc(p_norm_gated_fwd(o.data_ptr(), gate.data_ptr(), in[NW].data_ptr(), nullptr, nullptr, y.data_ptr(), nullptr, nullptr, (float*)rstd.data_ptr(),
                                  rows * HV, V, (float)eps, code, code_of(in[NW].scalar_type()), GDN_DTYPE_F32, GDN_DTYPE_F32, GDN_ACT_SILU, 1, stream), "gdn_norm_gated_fwd");
        const at::Tensor out = at::mm(y, in[OW].t()).view({B, T, in[OW].size(0)});
        variable_list keep(in.begin(), in.end());
        for (const at::Tensor& t : {w, p, gate, qkv[0], qkv[1], qkv[2], graw, braw, o, y, rstd}) keep.push_back(t);
        ctx->save_for_backward(keep);
        ctx->saved_data["heads"] = heads;
        ctx->saved_data["type"] = (int64_t)type;
        ctx->saved_data["device"] = dev;
        ctx->saved_data["neg"] = neg;
        return {out};
    }
    static ChunkCall call_of(int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V, bool neg) {
        return ChunkCall{B, T, H, HV, K, V, B, B * ((T + 63) / 64), std::pow((double)K, -0.5),
                         GDN_FLAG_QK_L2NORM | GDN_FLAG_BETA_SIGMOID | GDN_FLAG_STATE_V_FIRST | (neg ? GDN_FLAG_NEG_EIGVAL : 0u), false, true};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const c10::Device dev = ctx->saved_data["device"].toDevice();
        const c10::DeviceGuard guard(dev);
        const at::ScalarType type = (at::ScalarType)ctx->saved_data["type"].toInt();
        auto s = ctx->get_saved_variables();
        for (int i = 0; i < (int)s.size(); ++i)
            s[i] = saved(s[i], i >= A_LOG && i <= NW ? s[i].scalar_type() : i == INPUTS + 10 ? at::kFloat : type, dev);
        const at::Tensor &w = s[INPUTS], &p = s[INPUTS + 1], &gate = s[INPUTS + 2], *qkv = &s[INPUTS + 3], &graw = s[INPUTS + 6], &braw = s[INPUTS + 7],
                         &o = s[INPUTS + 8], &y = s[INPUTS + 9], &rstd = s[INPUTS + 10], &x = s[X];
        void* stream = stream_of(dev);
        const int code = code_of(type);
        const int64_t heads = ctx->saved_data["heads"].toInt();
        const bool neg = ctx->saved_data["neg"].toBool();
        const int64_t B = x.size(0), T = x.size(1), hidden = x.size(2), rows = B * T, kd = s[QW].size(0), vd = s[VW].size(0), HV = s[AW].size(0);
        const int64_t K = kd / heads, V = vd / HV, W = s[QC].size(-1), ld = w.size(0), used = 2 * kd + vd + 2 * HV;
        const at::Tensor dy = grads[0].to(type).reshape({rows, -1}), x2 = x.reshape({rows, hidden});
        variable_list r(INPUTS + 3);
        if (ctx->needs_input_grad(OW)) r[OW] = at::mm(dy.t(), y);
        const at::Tensor dyn = at::mm(dy, s[OW]);
        // the gated norm
        const at::Tensor dob = at::empty_like(o), dgate = at::empty_like(gate);
        const int64_t parts = std::max<int64_t>(1, std::min<int64_t>(1024, (rows * HV + 31) / 32));
        const at::Tensor dnw = empty_on(dev, at::kFloat, {parts, V});
        check_rc(p_norm_gated_bwd(dyn.data_ptr(), o.data_ptr(), gate.data_ptr(), s[NW].data_ptr(), nullptr, nullptr, (const float*)rstd.data_ptr(), nullptr,
                                  dob.data_ptr(), dgate.data_ptr(), (float*)dnw.data_ptr(), nullptr, rows * HV, V, V, parts, code,
                                  code_of(s[NW].scalar_type()), GDN_ACT_SILU, 1, stream), "gdn_norm_gated_bwd");
        r[NW] = sum_rows(dnw, s[NW].scalar_type(), s[NW].sizes(), stream);
        // the operator, then its gate and beta into their columns of the projections' gradient
        const at::Tensor A = to_f32(s[A_LOG]), dt = to_f32(s[DT]), none;
        const ChunkGrads c = chunk_backward(call_of(B, T, heads, HV, K, V, neg), qkv[0], qkv[1], qkv[2], graw.data_ptr(), braw.data_ptr(), code, A, dt, none,
                                            none, none, none, dob, none);
        const at::Tensor dp = empty_on(dev, type, {rows, ld});
        char* dpb = (char*)dp.data_ptr();
        const int64_t gp = gate_parts(rows, HV), col = 2 * kd + vd;
        const at::Tensor gpart = empty_on(dev, at::kFloat, {gp, 2, HV});
        check_rc(p_gate_bwd((const float*)c.dg.data_ptr(), (const float*)c.db.data_ptr(), graw.data_ptr(), braw.data_ptr(), (const float*)A.data_ptr(),
                            (const float*)dt.data_ptr(), dpb + col * 2, dpb + (col + HV) * 2, (float*)gpart.data_ptr(), rows, HV, gp, HV, HV, ld, ld,
                            2 * HV, ld - col, code, code, neg ? 2.f : 1.f, stream), "gdn_gate_bwd");
        const at::Tensor sums = sum_rows(gpart, s[A_LOG].scalar_type(), {2, HV}, stream);
        r[A_LOG] = sums[0]; r[DT] = sums[1];
        // the convolutions, each into its columns
        const at::Tensor dconv[3] = {c.dq, c.dk, c.dv};
        int64_t at = 0;
        for (int i = 0; i < 3; ++i) {
            const int64_t D = i < 2 ? kd : vd, tiles = B * ((T + 63) / 64), run = conv_bwd_run(tiles, D);
            const at::Tensor part = empty_on(dev, at::kFloat, {(tiles + run - 1) / run, D, W});
            check_rc(p_conv_bwd_runs((const char*)p.data_ptr() + at * 2, s[QC + i].data_ptr(), nullptr, nullptr, dconv[i].data_ptr(), nullptr, dpb + at * 2,
                                     (float*)part.data_ptr(), nullptr, nullptr, nullptr, nullptr, B, T, D, W, B, tiles, T * ld, ld, ld, run, code, code,
                                     GDN_DTYPE_F32, GDN_ACT_SILU, 0, stream), "gdn_causal_conv1d_bwd");
            r[QC + i] = sum_rows(part, type, s[QC + i].sizes(), stream);
            at += D;
        }
        // the projections
        if (ctx->needs_input_grad(X)) {
            at::Tensor dx = at::mm(dp, w);
            dx.addmm_(dgate.view({rows, vd}), s[GW]);
            r[X] = dx.view(x.sizes());
        }
        if (ctx->needs_input_grad(GW)) r[GW] = at::mm(dgate.view({rows, vd}).t(), x2);
        if (ctx->needs_input_grad({{QW, BW + 1}})) {
            const at::Tensor dw = at::mm(dp.t(), x2);
            at = 0;
            for (int i = QW; i <= BW; ++i) { r[i] = dw.narrow(0, at, s[i].size(0)); at += s[i].size(0); }
        }
        return r;
    }
};

// (x, q, k, v, a, b, g, o weights, (q, k, v conv weights [D,1,W]), A_log, dt_bias, norm weight, norm eps, neg_eigval, num_heads): the
// layer's forward on whole dense sequences without a cache.  None: not a call for the native path
PyObject* layer_train(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 15) { PyErr_SetString(PyExc_TypeError, "gdn_host.layer_train takes 15 arguments"); return nullptr; }
    variable_list in(LayerTrain::INPUTS);
    if (!PyTuple_Check(a[8]) || PyTuple_GET_SIZE(a[8]) != 3) Py_RETURN_NONE;
    PyObject* const src[LayerTrain::INPUTS] = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], PyTuple_GET_ITEM(a[8], 0), PyTuple_GET_ITEM(a[8], 1),
                                               PyTuple_GET_ITEM(a[8], 2), a[9], a[10], a[11]};
    for (int i = 0; i < LayerTrain::INPUTS; ++i) {
        const Arg t(src[i]);
        if (!t || !t->is_cuda()) Py_RETURN_NONE;
        in[i] = *t.t;
    }
    const at::Tensor& x = in[LayerTrain::X];
    const c10::Device dev = x.device();
    const at::ScalarType type = x.scalar_type();
    if ((type != at::kBFloat16 && type != at::kHalf) || x.dim() != 3 || x.numel() == 0 || dev.index() != c10::hip::current_device()) Py_RETURN_NONE;
    for (int i = 0; i < LayerTrain::INPUTS; ++i)
        if (in[i].device() != dev || !in[i].is_contiguous() || !aligned16(in[i].data_ptr()) || (i < LayerTrain::A_LOG && in[i].scalar_type() != type)) Py_RETURN_NONE;
    const int64_t hidden = x.size(2), heads = PyLong_AsLongLong(a[14]);
    const double eps = PyFloat_AsDouble(a[12]);
    if (PyErr_Occurred()) return nullptr;
    const int64_t kd = in[LayerTrain::QW].size(0), vd = in[LayerTrain::VW].size(0), HV = in[LayerTrain::AW].size(0);
    for (int i = LayerTrain::QW; i <= LayerTrain::GW; ++i)
        if (in[i].dim() != 2 || in[i].size(1) != hidden) Py_RETURN_NONE;
    if (heads < 1 || HV < 1 || HV % heads || kd % heads || vd % HV || in[LayerTrain::KW].size(0) != kd || in[LayerTrain::GW].size(0) != vd ||
        in[LayerTrain::BW].size(0) != HV || in[LayerTrain::OW].dim() != 2 || in[LayerTrain::OW].size(1) != vd || hidden % 8)
        Py_RETURN_NONE;
    const int64_t K = kd / heads, V = vd / HV, W = in[LayerTrain::QC].size(-1);
    if (!((K == 64 && V == 64) || (K == 128 && V == 128) || (K == 256 && V % 128 == 0)) || V > 2048 || W < 1 || W > 8) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i)
        if (in[LayerTrain::QC + i].numel() != (i < 2 ? kd : vd) * W || in[LayerTrain::QC + i].size(-1) != W) Py_RETURN_NONE;
    const at::Tensor &A = in[LayerTrain::A_LOG], &dt = in[LayerTrain::DT], &nw = in[LayerTrain::NW];
    if (A.dim() != 1 || dt.dim() != 1 || A.numel() != HV || dt.numel() != HV || A.scalar_type() != dt.scalar_type() || code_of(A.scalar_type()) < 0 ||
        nw.dim() != 1 || nw.numel() != V || code_of(nw.scalar_type()) < 0)
        Py_RETURN_NONE;
    const bool neg = truth(a[13]);
    variable_list r;
    {
        const NoGil free;
        r = LayerTrain::apply(at::TensorList(in), heads, neg, eps);
    }
    return THPVariable_Wrap(r[0]);
    END_HANDLE_TH_ERRORS
}
