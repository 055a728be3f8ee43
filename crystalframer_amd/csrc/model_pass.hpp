// Host side of cfh_model_forward / cfh_model_backward: the launches of a whole pass, one after the other, with every
// intermediate in the caller's arena.  Included by crystalframer_hip.hip behind the entry points it calls.
//
// What bounds a pass over a small batch is not any kernel but the host between them: the same launches made from Python,
// one autograd function per operator with its allocations, took 755 us per inference pass and 2330 us per training step
// against 168 and 515 us of kernels (4 layers, 1 and 13 crystals).
namespace {

struct ModelLayerBuffers {
    float *x1, *h, *qkv, *qs, *k, *v, *a;      // qkv .. a: inputs of this layer; x1, h: behind its core
    float *x2;                                 // output of this layer
    float *stream, *stream_bwd;                // weights of the bridge behind this layer's core in the order of their use
    float *frames, *z, *prob, *hist, *out, *wcat;
    uint32_t* records;
};
constexpr int MODEL_MAX_LAYERS = 64;
struct ModelBuffers {
    int64_t *edges, *e_start, *atom_start;
    int32_t* order;
    int4* heads;
    float *rpos, *recip, *rvlen, *vcell, *near_, *x0, *pooled;
    float4* table;
    char* geo_ws;
    float *front_stream, *front_stream_bwd;    // weights of the bridges in the order of their use
    float* y[CFH_MODEL_MAX_LINEARS];           // results of the head's linear layers but the last
    ModelLayerBuffers layer[MODEL_MAX_LAYERS];
    size_t total;
};
struct Carver {
    char* base;
    size_t off = 0;
    template <typename T>
    T* take(size_t n) {
        T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
        off += align256((n > 0 ? n : 1) * sizeof(T));
        return p;
    }
};

int check_model(const cfh_model* m, const cfh_model_batch* b) {
    if (!m || !b) return fail(CFH_EINVAL, "model and batch must not be NULL");
    if (m->struct_size != (int32_t)sizeof(cfh_model))
        return fail(CFH_EINVAL, "cfh_model.struct_size %d != %zu (header/library mismatch)", m->struct_size, sizeof(cfh_model));
    if (m->layers < 1 || m->layers > MODEL_MAX_LAYERS || !m->layer || !m->We)
        return fail(CFH_EINVAL, "model: 1 to %d layers with their weights and an embedding are needed", MODEL_MAX_LAYERS);
    if (m->heads < 1 || m->heads > 32 || m->D != m->heads * cfh::DH || m->D % 128 != 0 || 256 % m->D != 0 ||
        m->F < 128 || m->F % 128 != 0 || m->feat < 1 || m->feat > 512)
        return fail(CFH_EINVAL, "model: D=%d (16 x H=%d), F=%d, feat=%d not supported", m->D, m->heads, m->F, m->feat);
    if (m->linears < 1 || m->linears > CFH_MODEL_MAX_LINEARS)
        return fail(CFH_EINVAL, "model: %d linear layers in the head (1 to %d)", m->linears, CFH_MODEL_MAX_LINEARS);
    for (int i = 0; i < m->linears; i++) {
        const cfh_model_linear& T = m->head[i];
        if (!T.W || T.in % 16 != 0 || T.in != (i ? m->head[i - 1].out : m->D) || T.in > CFH_MODEL_MAX_WIDTH || T.out < 1 ||
            T.out > CFH_MODEL_MAX_WIDTH)
            return fail(CFH_EINVAL, "model: head layer %d (%d -> %d) not supported", i, T.in, T.out);
    }
    for (int l = 0; l < m->layers; l++) {
        const cfh_model_layer& L = m->layer[l];
        if (int rc = check_core_params(&L.core)) return rc;
        if (L.core.num_heads != m->heads || L.core.angle_bins != m->layer[0].core.angle_bins)
            return fail(CFH_EINVAL, "model: layer %d differs from layer 0 in heads or angle bins", l);
        if (!L.Wqkv || !L.bqkv || !L.lattice_w || !L.W_dist || !L.Wo || !L.bo || !L.W1 || !L.b1 || !L.W2 || !L.b2 ||
            (L.core.angle_bins > 0 && (!L.W_axis1 || !L.W_axis2 || !L.W_axis3)))
            return fail(CFH_EINVAL, "model: a weight of layer %d is NULL", l);
    }
    if (b->N < 1 || b->B < 1 || b->E < 1 || b->B > 0x7fffffffLL / 64)
        return fail(CFH_EINVAL, "model: N=%lld B=%lld E=%lld", (long long)b->N, (long long)b->B, (long long)b->E);
    return check_core_sizes(&m->layer[0].core, b->N, b->E);
}

// The tables of the geometry (sorted shifts, nearest images) are those of one half-width at a time: a layer that needs another
// one than the arena holds makes them again.
int layer_half_width(const cfh_model_layer& L) { return usual_half_width(&L.core, L.adaptive != 0); }
// What the arena holds before a backward pass: the half-width that all layers with tables share; -1 when they differ (the
// layers of the forward pass and of an earlier backward pass have then left one or the other).
int shared_half_width(const cfh_model* m) {
    int R = 0;
    for (int l = 0; l < m->layers; l++) {
        const int r = layer_half_width(m->layer[l]);
        if (r > 0 && R > 0 && r != R) return -1;
        if (r > 0) R = r;
    }
    return R;
}

// Layout of the arena.  keep: every layer its own buffers, for the backward pass; else the layers share one set (a layer
// reads its inputs before the next one's are written: the inputs of a layer alternate between two sets).
void model_buffers(const cfh_model* m, const cfh_model_batch* b, ModelBuffers& M) {
    Carver c{reinterpret_cast<char*>(b->arena)};
    const size_t N = b->N, E = b->E, B = b->B, D = m->D, F = m->F, H = m->heads;
    const int ang = m->layer[0].core.angle_bins;
    const size_t hw = cfh::core_hist_words(ang, !b->keep);
    M.edges = c.take<int64_t>(2 * E);
    M.e_start = c.take<int64_t>(N + 1);
    M.atom_start = c.take<int64_t>(B + 1);
    M.order = c.take<int32_t>(N);
    M.heads = c.take<int4>(2 * N);
    M.rpos = c.take<float>(3 * E);
    M.recip = c.take<float>(9 * B);
    M.rvlen = c.take<float>(3 * B);
    M.vcell = c.take<float>(B);
    M.geo_ws = c.take<char>((2 * B + 1) * sizeof(int64_t));
    M.table = c.take<float4>(B * cfh::FC_TCAP);
    M.near_ = c.take<float>(2 * E);
    M.x0 = c.take<float>(N * D);
    M.pooled = c.take<float>(B * D);
    // (a pass that keeps nothing has its own bridges, with streams of their own)
    M.front_stream = c.take<float>(b->keep ? bridge_stream_floats(cfh::BS_INPUTS, m->D, m->F, true, m->feat)
                                           : split_stream_floats(cfh::BS_INPUTS, m->D, m->F, true, m->feat));
    M.front_stream_bwd = b->keep ? c.take<float>(bridge_stream_floats(cfh::BS_INPUTS_BACKWARD, m->D, m->F, true)) : nullptr;
    for (int i = 0; i + 1 < m->linears; i++) M.y[i] = c.take<float>(B * (size_t)m->head[i].out);
    ModelLayerBuffers set[2];
    for (int l = 0; l < m->layers; l++) {
        ModelLayerBuffers& L = M.layer[l];
        const bool next = l + 1 < m->layers;
        float* const stream = c.take<float>(b->keep ? bridge_stream_floats(cfh::BS_FORWARD, m->D, m->F, next)
                                                    : split_stream_floats(cfh::BS_FORWARD, m->D, m->F, next));
        float* const stream_bwd = b->keep ? c.take<float>(bridge_stream_floats(cfh::BS_BACKWARD, m->D, m->F, next)) : nullptr;
        float* const wcat = c.take<float>(D * hw);
        if (b->keep || l < 2) {
            L.qs = c.take<float>(N * D); L.k = c.take<float>(N * D); L.v = c.take<float>(N * D); L.a = c.take<float>(N * H);
            L.x2 = c.take<float>(N * D);
            L.qkv = b->keep ? c.take<float>(N * 3 * D) : nullptr;
            if (b->keep || l == 0) {
                const bool split = infer_split(b->N, m->F);      // (the bridge in two launches passes its parts through memory)
                L.x1 = b->keep ? c.take<float>(N * D) : nullptr;
                L.h = b->keep ? c.take<float>(N * F) : (split ? c.take<float>(F / 128 * N * D) : nullptr);
                L.frames = c.take<float>(9 * N * H);
                if (b->keep) { L.z = c.take<float>(E * H); L.prob = c.take<float>(E * H); }
                // (inference in one launch per layer keeps the histograms in LDS)
                bool hist = b->keep != 0;
                for (int k = 0; k < m->layers; k++) hist |= !one_launch_form(&m->layer[k].core, b->N, b->E, ang > 0, true);
                L.hist = hist ? c.take<float>(H * (size_t)(b->keep || ang == 0 ? N : cfh::project_rows((int)N)) * hw) : nullptr;
                L.out = c.take<float>(N * D);
                L.records = c.take<uint32_t>(N * H * cfh::REC_WORDS);
            }
            if (l < 2) set[l] = L;
        }
        if (!b->keep && l > 0) {
            L = set[0];
            L.qs = set[l & 1].qs; L.k = set[l & 1].k; L.v = set[l & 1].v; L.a = set[l & 1].a; L.x2 = set[l & 1].x2;
        }
        L.stream = stream;
        L.stream_bwd = stream_bwd;
        L.wcat = wcat;
    }
    M.total = c.off;
    if (b->x0 && b->qkv0 && b->keep) {        // (only read)
        M.x0 = const_cast<float*>(b->x0);
        M.layer[0].qkv = const_cast<float*>(b->qkv0);
    }
}

// Rows of the per-block partial sums of a layer's lattice-weight gradient: the first layer's come from
// attention_inputs_bwd_kernel, the others' from the bridge.
int64_t model_partial_rows(const cfh_model* m, int l, int64_t N) {
    const int rows = l == 0 ? 4 * (256 / m->D) : 16;
    return (N + rows - 1) / rows;
}
struct ModelGrads {
    float *gx0, *gy[CFH_MODEL_MAX_LINEARS], *glogit, *gq, *gk, *gv, *ga;
    struct { float *g2, *gh, *g1, *g_attn, *gqkv, *gw_partial; } layer[MODEL_MAX_LAYERS];
    void* wgrad_ws;
    size_t wgrad_bytes, total;
};
size_t model_wgrad_bytes(const cfh_model* m, const cfh_model_batch* b);
void model_grads(const cfh_model* m, const cfh_model_batch* b, void* scratch, ModelGrads& G) {
    Carver c{reinterpret_cast<char*>(scratch)};
    const size_t N = b->N, E = b->E, B = b->B, D = m->D, F = m->F, H = m->heads;
    G.gx0 = c.take<float>(N * D);
    for (int i = 0; i < m->linears; i++) G.gy[i] = c.take<float>(B * (size_t)m->head[i].out);
    G.glogit = c.take<float>(E * H);
    G.gq = c.take<float>(N * D); G.gk = c.take<float>(N * D); G.gv = c.take<float>(N * D); G.ga = c.take<float>(N * H);
    for (int l = 0; l < m->layers; l++) {
        auto& L = G.layer[l];
        L.g2 = c.take<float>(N * D); L.gh = c.take<float>(N * F); L.g1 = c.take<float>(N * D);
        L.g_attn = c.take<float>(N * D); L.gqkv = c.take<float>(N * 3 * D);
        L.gw_partial = c.take<float>(model_partial_rows(m, l, b->N) * D);
    }
    G.wgrad_bytes = model_wgrad_bytes(m, b);
    G.wgrad_ws = c.take<char>(G.wgrad_bytes);
    G.total = c.off;
}

int64_t model_gradient_floats(const cfh_model* m) {
    const int64_t D = m->D, F = m->F, A = m->layer[0].core.angle_bins;
    int64_t n = D * m->feat + m->layers * (4 * D * D + 2 * D * F + D * (64 + 3 * A) + 3 * D + D + D + F + D);
    for (int i = 0; i < m->linears; i++) n += (int64_t)m->head[i].out * (m->head[i].in + 1);
    return n;
}

// The products that make the weight and bias gradients of the projections (pointers filled in from M, G and grads; with
// null buffers the list has the right sizes).
std::vector<cfh_linear_grad_job> model_wgrad_jobs(const cfh_model* m, const cfh_model_batch* b, const ModelBuffers& M,
                                                  const ModelGrads& G, float* grads, float** core_grads) {
    std::vector<cfh_linear_grad_job> jobs;
    const int64_t N = b->N, D = m->D, F = m->F, A = m->layer[0].core.angle_bins;
    float* g = grads;
    auto next = [&](int64_t n) { float* p = g; g += n; return p; };
    auto job = [&](const float* x, const float* dy, float* dW, float* db, int64_t rows, int64_t I, int64_t O) {
        jobs.push_back(cfh_linear_grad_job{x, dy, dW, db, rows, I, O, I, O});
    };
    job(b->x, G.gx0, next(D * m->feat), nullptr, N, m->feat, D);
    for (int l = 0; l < m->layers; l++) {
        const ModelLayerBuffers& L = M.layer[l];
        float* const gWqkv = next(3 * D * D);
        job(l ? M.layer[l - 1].x2 : M.x0, G.layer[l].gqkv, gWqkv, next(3 * D), N, D, 3 * D);
        float* const gWo = next(D * D);
        job(L.out, G.layer[l].g1, gWo, next(D), N, D, D);
        // (column sums of the per-block partial sums)
        jobs.push_back(cfh_linear_grad_job{nullptr, G.layer[l].gw_partial, nullptr, next(D), model_partial_rows(m, l, N), 1, D, 1, D});
        for (int e = 0; e < (A > 0 ? 4 : 1); e++) {
            float* const p = next(D * (e == 0 ? 64 : A));
            if (core_grads) core_grads[4 * l + e] = p;
        }
        float* const gW1 = next(F * D);
        job(L.x1, G.layer[l].gh, gW1, next(F), N, D, F);
        float* const gW2 = next(D * F);
        job(L.h, G.layer[l].g2, gW2, next(D), N, F, D);
    }
    for (int i = 0; i < m->linears; i++) {
        const cfh_model_linear& T = m->head[i];
        float* const gW = next((int64_t)T.out * T.in);
        job(i ? M.y[i - 1] : M.pooled, G.gy[i], gW, next(T.out), b->B, T.in, T.out);
    }
    return jobs;
}
// Which jobs of that list share the slicing of their rows.  With the 64-bin and without the angle encoding all of them
// (empty: one group); with the 16-bin encoding, whose small histograms leave the layers short, the jobs that become
// ready together while the pass walks down the layers, so that each group spreads over the whole chip.
std::vector<int32_t> model_wgrad_groups(const cfh_model* m) {
    std::vector<int32_t> g;
    const int L = m->layers;
    if (m->layer[0].core.angle_bins != cfh::SMALL_A) return g;
    g.push_back(L);                                          // embedding
    for (int l = 0; l < L; l++) {
        g.push_back(L - l);                                  // input projection
        g.push_back(L - 1 - l);                              // output projection
        g.push_back(L - l);                                  // lattice weights
        g.push_back(L - 1 - l);
        g.push_back(L - 1 - l);                              // feed-forward block
    }
    for (int i = 0; i < m->linears; i++) g.push_back(0);
    return g;
}
size_t model_wgrad_bytes(const cfh_model* m, const cfh_model_batch* b) {
    // (sizes and alignment are all that counts here: the pointers stand for the 256-byte aligned buffers of the pass)
    static float dummy;
    ModelBuffers M{};
    ModelGrads G{};
    std::vector<cfh_linear_grad_job> jobs = model_wgrad_jobs(m, b, M, G, nullptr, nullptr);
    float* d = reinterpret_cast<float*>(((uintptr_t)&dummy) & ~(uintptr_t)255);
    for (size_t j = 0; j < jobs.size(); j++) {
        // (distinct destinations: none of them overlap)
        if (jobs[j].I > 1 || jobs[j].x) jobs[j].x = d;
        const bool has_w = jobs[j].I > 1;
        jobs[j].dy = d;
        jobs[j].dW = has_w ? d + (j << 24) : nullptr;
        jobs[j].db = has_w ? nullptr : d + (j << 24);
    }
    if ((int)jobs.size() > cfh::WGRAD_MAX_JOBS)
        return cfh_linear_weight_bias_grad_batch_workspace_bytes(jobs.data(), (int32_t)jobs.size());
    const std::vector<int32_t> group = model_wgrad_groups(m);
    cfh::WgradJobs T;
    plan_wgrad(jobs.data(), 0, (int32_t)jobs.size(), T, group.empty() ? nullptr : group.data());
    return 256 + (size_t)T.blocks * cfh::WG_PART * sizeof(float);
}

void tail_args(const cfh_model* m, const cfh_model_batch* b, const ModelBuffers& M, cfh::TailArgs& T) {
    std::memset(&T, 0, sizeof(T));
    T.atom_start = M.atom_start; T.pooled = M.pooled;
    T.B = (int)b->B; T.D = m->D; T.nlin = m->linears;
    // (with 256 crystals and more every compute unit has a workgroup of its own already)
    T.per_wg = b->B <= 512 ? 1 : (b->B <= 2048 ? 4 : cfh::TAIL_ROWS);
    int widest = m->D;
    for (int i = 0; i < m->linears; i++) {
        cfh::TailLinear& L = T.lin[i];
        L.W = m->head[i].W; L.b = m->head[i].b; L.K = m->head[i].in; L.O = m->head[i].out; L.relu = m->head[i].relu;
        L.y = i + 1 < m->linears ? M.y[i] : nullptr;
        if (L.O > widest) widest = L.O;
    }
    T.ld = (widest + 3) / 4 * 4 + cfh::TAIL_PAD;
}
int tail_launch(const cfh::TailArgs& T, const float* gout, hipStream_t st) {
    const dim3 grid((unsigned)((T.B + T.per_wg - 1) / T.per_wg)), block(64 * cfh::TAIL_WAVES);
    const size_t lds = 2 * (size_t)cfh::TAIL_ROWS * T.ld * sizeof(float);
    TimedScope timed("model_tail", st);
    if (int rc = gout ? allow_lds<cfh::model_tail_bwd_kernel>(lds) : allow_lds<cfh::model_tail_fwd_kernel>(lds)) return rc;
    if (gout) hipLaunchKernelGGL(cfh::model_tail_bwd_kernel, grid, block, lds, st, T, gout);
    else hipLaunchKernelGGL(cfh::model_tail_fwd_kernel, grid, block, lds, st, T);
    return finish_launch("model_tail");
}
}  // namespace

extern "C" {

int64_t cfh_model_sizes(const cfh_model* m, const cfh_model_batch* b, size_t bytes[4]) try {
    if (int rc = check_model(m, b)) return rc;
    if (!bytes) return fail(CFH_EINVAL, "bytes must not be NULL");
    cfh_model_batch q = *b;
    q.arena = nullptr;
    ModelBuffers M{};
    model_buffers(m, &q, M);
    bytes[0] = M.total;
    bytes[1] = core_layout(&m->layer[0].core, b->N, b->E, b->B, false).total;
    bytes[2] = bytes[3] = 0;
    if (b->keep) {
        ModelGrads G{};
        model_grads(m, &q, nullptr, G);
        bytes[2] = G.total;
        bytes[3] = core_layout(&m->layer[0].core, b->N, b->E, b->B, true).total;
        const size_t wg = cfh_fused_core_weight_gradients_workspace_bytes(&m->layer[0].core, m->layers);
        if (wg > bytes[3]) bytes[3] = wg;
    }
    return model_gradient_floats(m);
} catch (const std::exception& e) {
    return fail(CFH_ELAUNCH, "model: %s", e.what());      // (host memory: nothing is thrown through a C entry point)
}

int cfh_model_forward(const cfh_model* m, const cfh_model_batch* b, float* out) try {
    int rc = check_model(m, b);
    if (rc) return rc;
    if (!b->x || !b->pos || !b->batch || !b->tvecs || !b->sizes || !out)
        return fail(CFH_EINVAL, "model: x, pos, batch, tvecs, sizes and out must not be NULL");
    ModelBuffers M{};
    model_buffers(m, b, M);
    if (!b->arena || b->arena_bytes < M.total || ((uintptr_t)b->arena & 255))
        return fail(CFH_EWORKSPACE, "model: arena of %zu bytes (256-byte aligned) needed, %zu given", M.total, b->arena_bytes);
    hipStream_t st = (hipStream_t)b->stream;
    const int64_t N = b->N, E = b->E, B = b->B;
    const int D = m->D, F = m->F, H = m->heads;
    TimedScope whole("model_forward", st);
    // the weights of the bridges in the order of their use, the cores' concatenated weights, the geometry
    {
        TimedScope timed("model_start", st);
        cfh::StartArgs A{};
        cfh::GeometryArgs& g = A.geo;
        g.pos = b->pos; g.batch = b->batch; g.tvecs = b->tvecs; g.sizes = b->sizes;
        g.edges = M.edges; g.rpos = M.rpos; g.recip = M.recip; g.rvlen = M.rvlen; g.vcell = M.vcell;
        g.e_start = M.e_start; g.order = M.order; g.heads = M.heads; g.atom_start = M.atom_start;
        g.pair_start = reinterpret_cast<int64_t*>(M.geo_ws);
        g.order_start = g.pair_start + (B + 1);
        g.N = (int32_t)N; g.B = (int32_t)B; g.E = E;
        A.geo_blocks = 2;
        A.table_R = layer_half_width(m->layer[0]);
        if (A.table_R > 0) {
            constexpr int per = cfh::START_THREADS / cfh::FC_TCAP;
            A.table = M.table;
            A.table_blocks = (int)((B + per - 1) / per);
        }
        StreamList S(D, F, st, m->feat, !b->keep);
        S.add(cfh::BS_INPUTS, m->We, nullptr, nullptr, m->layer[0].Wqkv, M.front_stream);
        if (b->keep) S.add(cfh::BS_INPUTS_BACKWARD, nullptr, nullptr, nullptr, m->layer[0].Wqkv, M.front_stream_bwd);
        cfh::StartWcat W{};
        W.hc = H * cfh::DH;
        auto launch = [&]() {      // (also when the list of the streams is full)
            A.streams = S.T;
            const int stream_blocks = (S.blocks + cfh::START_THREADS / 256 - 1) / (cfh::START_THREADS / 256);
            hipLaunchKernelGGL(cfh::model_start_kernel, dim3((unsigned)(A.geo_blocks + A.table_blocks + stream_blocks)),
                               dim3(cfh::START_THREADS), 0, st, A);
            S.clear();
            A.geo_blocks = A.table_blocks = 0;
        };
        for (int l = 0; l < m->layers; l++) {
            const cfh_model_layer& L = m->layer[l];
            const cfh_params& p = L.core;
            const float* const Wq = l + 1 < m->layers ? m->layer[l + 1].Wqkv : nullptr;
            if (S.T.n + 2 > cfh::BR_MAX_STREAMS) launch();
            S.add(cfh::BS_FORWARD, L.Wo, L.W1, L.W2, Wq, M.layer[l].stream);
            if (b->keep) S.add(cfh::BS_BACKWARD, L.Wo, L.W1, L.W2, Wq, M.layer[l].stream_bwd);
            const bool ang = p.angle_bins > 0;
            const cfh::WcatArgs w{L.W_dist, ang ? L.W_axis1 : nullptr, ang ? L.W_axis2 : nullptr, ang ? L.W_axis3 : nullptr,
                                  cfh::core_hist_words(p.angle_bins, !b->keep), p.dist_coef, p.angle_coef, p.angle_wscale,
                                  M.layer[l].wcat};
            if (W.n < cfh::START_MAX_WCAT) W.w[W.n++] = w;
            else hipLaunchKernelGGL(cfh::core_wcat_kernel, dim3((unsigned)W.hc), dim3(256), 0, st, w);
        }
        launch();
        const int atom_blocks = (int)((N + 256) / 256);
        const cfh::PairsArgs P{g, A.table, reinterpret_cast<float2*>(M.near_), A.table_R, atom_blocks};
        hipLaunchKernelGGL(cfh::model_pairs_kernel, dim3((unsigned)(W.n * W.hc + atom_blocks + (E + 31) / 32)), dim3(256), 0, st, P, W);
        if ((rc = finish_launch("model_start"))) return rc;
    }
    {   // embedding and the inputs of the first layer
        const cfh_model_layer& L = m->layer[0];
        const ModelLayerBuffers& Y = M.layer[0];
        if (b->x0 && b->qkv0) {
            if (!b->keep) return fail(CFH_EINVAL, "model: x0 and qkv0 are taken with keep only");
            if ((rc = cfh_attention_inputs_forward(Y.qkv, L.lattice_w, L.gauss_scale_dev, L.c1, L.lb, L.c2, L.q_scale, N, H,
                                                   cfh::DH, Y.qs, Y.k, Y.v, Y.a, b->stream)))
                return rc;
        } else {
            cfh::BridgeArgs A{};
            A.attn = b->x; A.x2 = M.x0; A.feat = m->feat;
            A.stream = M.front_stream;
            A.steps = b->keep ? cfh::bridge_stream_steps(cfh::BS_INPUTS, D, F, true, m->feat)
                              : cfh::split_stream_steps(cfh::BS_INPUTS, D, F, true, m->feat);
            A.bq = L.bqkv; A.lattice_w = L.lattice_w; A.gauss = L.gauss_scale_dev;
            A.qkv = Y.qkv; A.qs = Y.qs; A.k = Y.k; A.v = Y.v; A.a = Y.a;
            A.N = (int)N; A.D = D; A.F = F; A.H = H;
            A.c1 = L.c1; A.lb = L.lb; A.c2 = L.c2; A.q_scale = L.q_scale;
            if ((rc = b->keep ? bridge_front(A, D, st) : front_infer(A, D, st))) return rc;
        }
    }
    int held = layer_half_width(m->layer[0]);
    for (int l = 0; l < m->layers; l++) {
        const cfh_model_layer& L = m->layer[l];
        const ModelLayerBuffers& Y = M.layer[l];
        cfh_params p = L.core;
        if (b->noise_seeds) p.noise_seed = b->noise_seeds[l];
        const int R = layer_half_width(L);
        const bool ready = R == held;
        if (R > 0) held = R;
        const cfh_core_cache cache{reinterpret_cast<float*>(M.table), M.near_, Y.wcat, Y.records, ready ? 1 : 0, 0, 0, 0};
        const bool ang = p.angle_bins > 0;
        if ((rc = fused_core_forward_impl(&p, Y.qs, Y.k, Y.v, Y.a, M.rpos, b->tvecs, L.adaptive ? M.rvlen : nullptr, b->batch,
                                         M.edges, M.e_start, M.order, L.W_dist, ang ? L.W_axis1 : nullptr,
                                         ang ? L.W_axis2 : nullptr, ang ? L.W_axis3 : nullptr, N, E, B,
                                         ang ? Y.frames : nullptr, ang ? 1 : 0, Y.z, Y.prob, Y.hist, Y.out, &cache,
                                         b->workspace, b->workspace_bytes, b->stream, !b->keep, true, M.heads)))
            return rc;
        const bool next = l + 1 < m->layers;
        const cfh_model_layer& Ln = m->layer[next ? l + 1 : l];
        const ModelLayerBuffers& Yn = M.layer[next ? l + 1 : l];
        cfh::BridgeArgs A{};
        A.attn = Y.out; A.xres = l ? M.layer[l - 1].x2 : M.x0;
        A.bo = L.bo; A.b1 = L.b1; A.b2 = L.b2;
        A.stream = Y.stream;
        A.steps = b->keep ? cfh::bridge_stream_steps(cfh::BS_FORWARD, D, F, next) : cfh::split_stream_steps(cfh::BS_FORWARD, D, F, next);
        A.x1 = Y.x1; A.h = Y.h; A.x2 = Y.x2;
        A.N = (int)N; A.D = D; A.F = F; A.H = H;
        if (next) {
            A.bq = Ln.bqkv; A.lattice_w = Ln.lattice_w; A.gauss = Ln.gauss_scale_dev;
            A.qkv = Yn.qkv; A.qs = Yn.qs; A.k = Yn.k; A.v = Yn.v; A.a = Yn.a;
            A.c1 = Ln.c1; A.lb = Ln.lb; A.c2 = Ln.c2; A.q_scale = Ln.q_scale;
        }
        if ((rc = b->keep ? bridge_forward(A, D, st) : bridge_infer(A, D, st))) return rc;
    }
    cfh::TailArgs T;
    tail_args(m, b, M, T);
    T.x = M.layer[m->layers - 1].x2;
    T.lin[m->linears - 1].y = out;
    return tail_launch(T, nullptr, st);
} catch (const std::exception& e) {
    return fail(CFH_ELAUNCH, "model forward: %s", e.what());
}

int cfh_model_backward(const cfh_model* m, const cfh_model_batch* b, const float* gout, void* scratch,
                       size_t scratch_bytes, float* grads) try {
    int rc = check_model(m, b);
    if (rc) return rc;
    if (!b->x || !b->pos || !b->batch || !b->tvecs || !b->sizes || !gout || !grads || !b->keep)
        return fail(CFH_EINVAL, "model backward: the forward's inputs (with keep), gout and grads must not be NULL");
    ModelBuffers M{};
    model_buffers(m, b, M);
    if (!b->arena || b->arena_bytes < M.total || ((uintptr_t)b->arena & 255))
        return fail(CFH_EWORKSPACE, "model: arena of %zu bytes (256-byte aligned) needed, %zu given", M.total, b->arena_bytes);
    ModelGrads G{};
    model_grads(m, b, scratch, G);
    if (!scratch || scratch_bytes < G.total || ((uintptr_t)scratch & 255))
        return fail(CFH_EWORKSPACE, "model: scratch of %zu bytes (256-byte aligned) needed, %zu given", G.total, scratch_bytes);
    if (m->head[m->linears - 1].relu) return fail(CFH_EINVAL, "model: a rectifier behind the last linear layer");
    hipStream_t st = (hipStream_t)b->stream;
    const int64_t N = b->N, E = b->E, B = b->B;
    const int D = m->D, F = m->F, H = m->heads;
    TimedScope whole("model_backward", st);
    cfh::TailArgs T;
    tail_args(m, b, M, T);
    for (int i = 0; i < m->linears; i++) T.lin[i].gy = G.gy[i];
    T.gx = G.layer[m->layers - 1].g2;
    if ((rc = tail_launch(T, gout, st))) return rc;

    int held = shared_half_width(m);
    for (int l = m->layers - 1; l >= 0; l--) {
        // the projections between the core of layer l and the inputs of layer l + 1
        const cfh_model_layer& L = m->layer[l];
        const ModelLayerBuffers& Y = M.layer[l];
        auto& g = G.layer[l];
        const bool next = l + 1 < m->layers;
        cfh::BridgeBwdArgs A{};
        A.h = Y.h; A.stream = Y.stream_bwd; A.steps = cfh::bridge_stream_steps(cfh::BS_BACKWARD, D, F, next);
        A.g_x2 = next ? G.layer[l + 1].g1 : g.g2;
        A.g2 = g.g2; A.gh = g.gh; A.g1 = g.g1; A.g_attn = g.g_attn;
        A.N = (int)N; A.F = F; A.H = H;
        A.klen_q = bridge_klen(3 * D, D);
        if (next) {
            const cfh_model_layer& Ln = m->layer[l + 1];
            A.ai_qkv = M.layer[l + 1].qkv; A.ai_w = Ln.lattice_w; A.ai_gauss = Ln.gauss_scale_dev;
            A.ai_gqs = G.gq; A.ai_gk = G.gk; A.ai_gv = G.gv; A.ai_ga = G.ga;
            A.gqkv_out = G.layer[l + 1].gqkv; A.gw_partial = G.layer[l + 1].gw_partial;
            A.c1 = Ln.c1; A.lb = Ln.lb; A.c2 = Ln.c2; A.q_scale = Ln.q_scale;
        }
        if ((rc = bridge_backward(A, D, st))) return rc;
        cfh_params p = L.core;
        p.flags |= CFH_FLAG_NO_WEIGHT_GRADS;
        const int R = layer_half_width(L);
        const bool table_ready = R == held;
        if (R > 0) held = R;
        const cfh_core_cache cache{reinterpret_cast<float*>(M.table), nullptr, Y.wcat, Y.records, table_ready ? 1 : 0, 1, 1, 0};
        const bool ang = p.angle_bins > 0;
        if ((rc = fused_core_backward_impl(&p, Y.qs, Y.k, Y.v, Y.a, M.rpos, b->tvecs, L.adaptive ? M.rvlen : nullptr, b->batch,
                                          M.edges, M.e_start, M.order, L.W_dist, ang ? L.W_axis1 : nullptr,
                                          ang ? L.W_axis2 : nullptr, ang ? L.W_axis3 : nullptr, ang ? Y.frames : nullptr, Y.z,
                                          Y.prob, Y.hist, Y.out, G.layer[l].g_attn, N, E, B, G.gq, G.gk, G.gv, G.ga, G.glogit,
                                          nullptr, nullptr, nullptr, nullptr, &cache, b->workspace, b->workspace_bytes,
                                          b->stream, true)))
            return rc;
    }
    {   // the inputs of the first layer: gradient of its projection, of the embedded atoms (projection + residual)
        const cfh_model_layer& L = m->layer[0];
        auto& g = G.layer[0];
        if ((rc = cfh_attention_inputs_backward(M.layer[0].qkv, L.lattice_w, L.gauss_scale_dev, L.c1, L.lb, L.c2, L.q_scale, G.gq,
                                                G.gk, G.gv, G.ga, N, H, cfh::DH, g.gqkv, nullptr, g.gw_partial,
                                                (size_t)model_partial_rows(m, 0, N) * D * sizeof(float), b->stream)))
            return rc;
        cfh::BridgeBwdArgs A{};
        A.g_x2 = g.g1; A.gqkv = g.gqkv; A.g2 = G.gx0;
        A.stream = M.front_stream_bwd; A.steps = cfh::bridge_stream_steps(cfh::BS_INPUTS_BACKWARD, D, F, true);
        A.N = (int)N; A.F = F; A.H = H;
        A.inputs_only = 1;
        A.klen_q = 3 * D;                      // (one sum, as small_linear_dx_kernel makes it)
        if ((rc = bridge_backward(A, D, st))) return rc;
    }
    // the weight gradients of the whole pass: the projections, then the cores
    std::vector<float*> core_grads(4 * (size_t)m->layers, nullptr);
    const std::vector<cfh_linear_grad_job> jobs = model_wgrad_jobs(m, b, M, G, grads, core_grads.data());
    const std::vector<int32_t> group = model_wgrad_groups(m);
    {
        TimedScope timed("linear_weight_gradients", st);
        if ((rc = linear_wgrad_batch_impl(jobs.data(), (int32_t)jobs.size(), G.wgrad_ws, G.wgrad_bytes, b->stream, true,
                                          group.empty() ? nullptr : group.data())))
            return rc;
    }
    std::vector<cfh_core_wgrad_job> cj;
    for (int l = 0; l < m->layers; l++) {
        cj.push_back(cfh_core_wgrad_job{G.layer[l].g_attn, M.layer[l].hist, N, core_grads[4 * l], core_grads[4 * l + 1],
                                        core_grads[4 * l + 2], core_grads[4 * l + 3]});
        // (layers whose encodings have the same constants go together)
        const bool last = l + 1 == m->layers;
        const cfh_params &p = m->layer[l].core, &q = m->layer[last ? l : l + 1].core;
        if (last || p.dist_coef != q.dist_coef || p.angle_coef != q.angle_coef || p.angle_wscale != q.angle_wscale) {
            if ((rc = core_weight_gradients_impl(&p, cj.data(), (int32_t)cj.size(), b->workspace, b->workspace_bytes, b->stream,
                                                 true)))
                return rc;
            cj.clear();
        }
    }
    return CFH_OK;
} catch (const std::exception& e) {
    return fail(CFH_ELAUNCH, "model backward: %s", e.what());
}

}  // extern "C"
