// resident_decode.hpp -- LPP_PATH_PERSISTENT for models whose layers fit an XCD: one kernel per token (included by
// dataflow_decode.hip, whose hand-overs, sampler and step record it shares).
//
// A model of a few million parameters has nothing to stream: at the 15M shape (dim 288, hidden 768, six layers, fp32) a
// layer's matrices are 4 MB, 0.6 us of HBM time, and k_decode_dataflow's token is 125 us of hand-overs between 256 compute
// units, 17.5 us a layer, while every phase has one or two rows for a streaming wavefront.  Here layer l belongs to XCD
// l % n_xcc alone.  Its 32 workgroups hold the layer's four matrices in REGISTERS, requested when the kernel starts (the
// layers of all XCDs at once) or when the XCD is done with the layer before, so a phase is a few multiply-adds between
// registers and LDS and a hand-over that stays in one L2 with nothing queued in front of it; only x crosses from the XCD
// of one layer to that of the next.  The first n_heads workgroups of an XCD hold the attention items, one query head each
// with its whole context in registers, the others share the rows.  The classifier's rows, dealt out over all workgroups
// of the device, wait in LDS by the time the last layer is done.
//
// What bounds it: latency.  Per layer five hand-overs of 0.8 to 1.2 us (four inside an XCD, one across) and the barriers
// and reductions between them.  15M shape, a token: 122 us before, 58 now: about 7 a layer, 6 the sampler.
//
// Every value is formed by exactly one workgroup; sums run over a lane's elements in order, then across the lanes.

constexpr int kResThreads = 1024;
constexpr int kResGroup = 16;         // lanes that share a row of dim columns: 64 rows to a workgroup and pass
constexpr int kResDimLoads = 5;       // 16-byte loads of such a lane: dim up to 320
constexpr int kResHiddenLoads = 3;    // the same of a whole wavefront on a row of hidden columns: hidden up to 768
constexpr int kResDim = kResGroup * 4 * kResDimLoads, kResHidden = kWave * 4 * kResHiddenLoads;
constexpr int kResPositions = 512;    // contexts whose K and V rows the registers of a workgroup hold (heads of up to 64)
constexpr int kResHead = 64;

struct Resident {
    u64* near;           // [n_xcc][3 * near_stride]: attention output, x behind the O projection, x behind the last layer
    int near_stride;
    int qkv, o, gu, down;  // rows (hidden units) of a row workgroup: blocks of the stacked [Wq; Wk; Wv], Wo, W1 / W3, W2
    int cls_in_lds;        // classifier rows of a workgroup that wait in LDS
};

// LDS and barrier only: __syncthreads would also wait for every global request, the weights on their way among them.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The value in a slot once it carries the wanted sequence number.
template <bool kNear>
__device__ __forceinline__ float await_value(const u64* slot, unsigned want, const Ctx& c) {
    u64 got;
    unsigned spins = 0;
    while (true) {
        got = kNear ? peek_near(slot) : peek(slot);
        if (tag_of(got) == want || poll_give_up(c, spins)) break;
    }
    return value_of(got);
}

// A lane's part of one row: 16-byte pieces lane + kLanes k, zeros past the row's end.
template <int kLoads, int kLanes>
__device__ __forceinline__ void request_row(floatx4 (&w)[kLoads], const float* row, int lane, int cols, bool exists) {
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
        const int col = 4 * (lane + kLanes * k);
        w[k] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        if (exists && col < cols) w[k] = *reinterpret_cast<const floatx4*>(row + col);
    }
}
template <int kLoads>
__device__ __forceinline__ float lane_dot(const floatx4 (&w)[kLoads], const floatx4 (&x)[kLoads]) {
    float part[2] = {0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kLoads; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[k & 1] = fmaf(w[k][e], x[k][e], part[k & 1]);
    return part[0] + part[1];
}
// (xs is zero past the vector's end)
template <int kLoads, int kLanes>
__device__ __forceinline__ float lane_dot(const floatx4 (&w)[kLoads], const float* xs, int lane) {
    floatx4 x[kLoads];
#pragma unroll
    for (int k = 0; k < kLoads; ++k) x[k] = *reinterpret_cast<const floatx4*>(xs + 4 * (lane + kLanes * k));
    return lane_dot(w, x);
}

// What the workgroup keeps in LDS besides its classifier rows.
struct ResidentLds {
    float* xraw;   // [kResDim] x as received; zero past dim
    float* xs;     // [kResDim] times the norm gain
    float* wide;   // [kResHidden] attention output or SwiGLU output; zero past their ends
    float* qkv;    // [kResHead] this token's q of the head, [2][kResHead] its k and v in binary16
    float* score;  // [kResPositions]
    float* part;   // [16][kResHead] wavefronts' weighted values
    float* cls;    // [cls_in_lds][dim]
};

// One query head: its context in registers before q arrives, a lane per quarter of a K row and a lane per 8 dimensions
// of a V row (model.cpp:186-198, softmax ops.cpp:56-75; the current position's k and v rounded as the cache holds them).
__device__ __forceinline__ void resident_attention(Ctx& c, const ResidentLds& l, const Resident& rs, int layer, int h) {
    const DecodeArgs& a = c.a;
    int tid = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tid), "+s"(h));
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int hs = a.head_size, pieces = hs >> 3, pos = c.pos, npos = pos + 1, kvh = h / a.gqa;
    const size_t head = (static_cast<size_t>(layer) * a.n_kv_heads + kvh) * a.seq_len * hs;
    const uintx4 none = uintx4{0u, 0u, 0u, 0u};
    constexpr int kPasses = kResPositions / 256, kRows = kResPositions / 128;
    uintx4 k[kPasses][2], v[kRows];
#pragma unroll
    for (int p = 0; p < kPasses; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = 256 * p + (tid >> 2), piece = (tid & 3) + 4 * j;
            k[p][j] = none;
            if (t < pos && piece < pieces) k[p][j] = load16(a.key_cache + head + static_cast<size_t>(t) * hs + 8 * piece);
        }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int t = 128 * r + (tid >> 3), piece = tid & 7;
        v[r] = none;
        if (t < pos && piece < pieces) v[r] = load16(a.value_cache + head + static_cast<size_t>(t) * hs + 8 * piece);
    }
    const u64* in = c.t.near_qkv + static_cast<size_t>(c.xcc) * c.t.near_qkv_stride;
    const unsigned tag = c.seq(layer, kQkv);
    half_t* current = reinterpret_cast<half_t*>(l.qkv + kResHead);  // k, then v of the current position
    if (tid < 3 * kResHead) {
        const int which = tid / kResHead, e = tid % kResHead;
        float got = 0.0f;
        if (e < hs) got = await_value<true>(in + (which == 0 ? h * hs : a.dim + (which - 1) * a.kv_dim + kvh * hs) + e, tag, c);
        if (which == 0) l.qkv[e] = got;
        else current[tid - kResHead] = static_cast<half_t>(got);
    }
    lds_barrier();
    // (only what the context reaches is worked through: the branches are the workgroup's)
    float q[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) q[j][e] = l.qkv[8 * ((tid & 3) + 4 * j) + e];
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        if (256 * p >= npos) break;
        const int t = 256 * p + (tid >> 2);
        if (t == pos) {
#pragma unroll
            for (int j = 0; j < 2; ++j) k[p][j] = *reinterpret_cast<const uintx4*>(current + 8 * ((tid & 3) + 4 * j));
        }
        float s[2] = {0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const half8_t kh = as_half8(k[p][j]);
#pragma unroll
            for (int e = 0; e < 8; ++e) s[j] = fmaf(static_cast<float>(kh[e]), q[j][e], s[j]);
        }
        float sum = s[0] + s[1];
        sum += dpp_move<kDppXor1>(sum);
        sum += dpp_move<kDppXor2>(sum);
        if ((tid & 3) == 0) l.score[t] = t < npos ? sum * c.t.inv_sqrt_head : -INFINITY;
    }
    lds_barrier();
    // every wavefront works out the maximum and the sum for itself: no barrier
    float top = -INFINITY, sum = 0.0f, mine[kResPositions / kWave];
#pragma unroll
    for (int i = 0; i < kResPositions / kWave; ++i) {
        if (kWave * i >= npos) break;
        mine[i] = l.score[kWave * i + lane];
        top = fmaxf(top, mine[i]);
    }
    top = wave_max(top);
#pragma unroll
    for (int i = 0; i < kResPositions / kWave; ++i) {
        if (kWave * i >= npos) break;
        sum += exp_fast(mine[i] - top);
    }
    sum = wave_sum(sum);
    float out[8] = {};
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        if (128 * r >= npos) break;
        const int t = 128 * r + (tid >> 3);
        if (t == pos) v[r] = *reinterpret_cast<const uintx4*>(current + kResHead + 8 * (tid & 7));
        const float w = exp_fast(l.score[t] - top);
        const half8_t vh = as_half8(v[r]);
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = fmaf(static_cast<float>(vh[e]), w, out[e]);
    }
    // (the eight lanes of a wavefront that hold the same dimensions)
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = congruent_sum<8>(out[e]);
    if (lane < 8) {
#pragma unroll
        for (int e = 0; e < 8; ++e) l.part[wave * kResHead + 8 * lane + e] = out[e];
    }
    lds_barrier();
    if (tid < hs) {
        float o = 0.0f;
#pragma unroll
        for (int w = 0; w < kResThreads / kWave; ++w) o += l.part[w * kResHead + tid];
        publish_near(rs.near + static_cast<size_t>(c.xcc) * 3 * rs.near_stride + h * hs + tid, o / sum, c.seq(layer, kAtt));
    }
    lds_barrier();  // (the areas are free for a later layer)
}

// 1 / sqrt(mean(xraw^2) + 1e-5), worked out by every wavefront for itself
__device__ __forceinline__ float resident_scale(const Ctx& c, const float* xraw) {
#pragma clang fp contract(off)
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < kResDim / kWave; ++k) {
        const float v = xraw[kWave * k + lane_id()];
        ss += v * v;
    }
    ss = wave_sum(ss);
    ss /= c.b.dim_as_float;
    ss += 1e-5f;
    return 1.0f / sqrtf(ss);
}

// Rows first .. first + n - 1 of `rows` for row workgroup w of blocks of `block` rows: how many there are.
__device__ __forceinline__ int resident_rows(int rows, int block, int w) {
    const int n = rows - w * block;
    return n < 0 ? 0 : (n > block ? block : n);
}

// The rows of one layer that row workgroup w owns (model.cpp:162-226).  then() is called behind the layer's requests.  (A
// workgroup without rows of a product does not wait for its inputs: nobody would wait for it in turn, and the slots may
// have gone on to a later layer by then.)
template <bool kGiven, class Then>
__device__ __forceinline__ void resident_rows_of_layer(Ctx& c, const ResidentLds& l, const Resident& rs, int layer, int w, Then then) {
#pragma clang fp contract(off)
    const DecodeArgs& a = c.a;
    // (opaque: what follows from these would otherwise be worked out ahead of the layer loop and held in registers)
    int tid = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tid), "+s"(w));
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int dim = a.dim, hidden = a.hidden, kv = a.kv_dim, hs = a.head_size, L = a.n_layers;
    const int n_qkv = resident_rows(dim + 2 * kv, rs.qkv, w), n_o = resident_rows(dim, rs.o, w);
    const int n_gu = resident_rows(hidden, rs.gu, w), n_down = resident_rows(dim, rs.down, w);
    const int group = lane >> 4, l16 = lane & 15, slot = 4 * wave + group;  // 64 row slots
    const int g = w * rs.qkv + slot;                                       // row of the stacked [Wq; Wk; Wv]
    floatx4 w_qkv[kResDimLoads], w_o[kResDimLoads], w_gu[kResDimLoads], w_down[kResHiddenLoads];
    {
        const char* m = g < dim ? a.wq : g < dim + kv ? a.wk : a.wv;
        const size_t row = g < dim ? static_cast<size_t>(layer) * dim + g : static_cast<size_t>(layer) * kv + (g < dim + kv ? g - dim : g - dim - kv);
        request_row<kResDimLoads, kResGroup>(w_qkv, reinterpret_cast<const float*>(m) + row * dim, l16, dim, slot < n_qkv);
    }
    auto request_rest = [&]() {
        request_row<kResDimLoads, kResGroup>(w_o, reinterpret_cast<const float*>(a.wo) + (static_cast<size_t>(layer) * dim + w * rs.o + slot) * dim, l16, dim,
                                             slot < n_o);
        request_row<kResDimLoads, kResGroup>(w_gu, reinterpret_cast<const float*>((slot & 1) ? a.w3 : a.w1) +
                                                       (static_cast<size_t>(layer) * hidden + w * rs.gu + (slot >> 1)) * dim,
                                             l16, dim, slot < 2 * n_gu);
        request_row<kResHiddenLoads, kWave>(w_down, reinterpret_cast<const float*>(a.w2) + (static_cast<size_t>(layer) * dim + w * rs.down + wave) * hidden,
                                            lane, hidden, wave < n_down);
    };
    // (the first layer cannot start before its q, k and v weights are in, and what is requested comes in in order: the
    // others' follow once those are out, and arrive while the attention items run)
    if (layer > 0) request_rest();
    then();
    u64* near = rs.near + static_cast<size_t>(c.xcc) * 3 * rs.near_stride;

    // q, k, v
    const int rotated = g < dim ? g : g - dim;  // RoPE pairs (2i, 2i + 1) sit in neighbouring lane groups
    const int within = rotated - div_head_size(c, rotated) * hs;
    const bool rotates = slot < n_qkv && g < dim + kv;
    // (requested ahead of the polls that wait for x, and in by then)
    float cos_t, sin_t;
    pinned_load(a.rope + static_cast<size_t>(c.pos) * (hs / 2) + (rotates ? within >> 1 : 0), cos_t, sin_t);
    if (n_qkv > 0 || n_o > 0) {
        if (tid < dim) {
            const float gain_att = pinned_load(a.rms_att + static_cast<size_t>(layer) * dim + tid);
            const float x = layer == 0 ? a.emb[static_cast<size_t>(c.token) * dim + tid] : await_value<false>(c.t.x + tid, c.seq(layer - 1, kDown), c);
            l.xraw[tid] = x;
            l.xs[tid] = x * gain_att;
        }
        lds_barrier();
    }
    if (n_qkv > 0) {
        const float scale = resident_scale(c, l.xraw);
        const float mine = row16_sum(lane_dot<kResDimLoads, kResGroup>(w_qkv, l.xs, l16)) * scale;
        const float other = lane_xor(mine, 16, lane);
        if (l16 == 0 && slot < n_qkv) {
            const float out = !rotates ? mine : (g & 1) ? other * sin_t + mine * cos_t : mine * cos_t - other * sin_t;
            publish_near(c.t.near_qkv + static_cast<size_t>(c.xcc) * c.t.near_qkv_stride + g, out, c.seq(layer, kQkv));
            if (g >= dim) {  // model.cpp:171-176
                const bool is_k = g < dim + kv;
                const int i = is_k ? g - dim : g - dim - kv;
                const int head = div_head_size(c, i);
                (is_k ? a.key_cache : a.value_cache)[((static_cast<size_t>(layer) * a.n_kv_heads + head) * a.seq_len + c.pos) * hs + (i - head * hs)] =
                    f32_to_f16_bits(out);
                if (layer == L - 1) (is_k ? a.k : a.v)[i] = out;
            } else if (layer == L - 1) {  // (the run state holds the last layer's: other XCDs write theirs to other L2s)
                a.q[g] = out;
            }
        }
    }
    if (kGiven && layer == L - 1) return;
    if (layer == 0) request_rest();
    // x + Wo . attention
    if (n_o > 0) {
        if (tid < dim) l.wide[tid] = await_value<true>(near + tid, c.seq(layer, kAtt), c);
        lds_barrier();
        const float sum = row16_sum(lane_dot<kResDimLoads, kResGroup>(w_o, l.wide, l16));
        const int row = w * rs.o + slot;
        if (l16 == 0 && slot < n_o) publish_near(near + rs.near_stride + row, l.xraw[row] + sum, c.seq(layer, kOproj));
        lds_barrier();  // (xraw is read before the next phase writes it)
    }
    // SwiGLU(W1 x, W3 x)
    if (n_gu > 0 || n_down > 0) {
        if (tid < dim) {
            const float gain_ffn = pinned_load(a.rms_ffn + static_cast<size_t>(layer) * dim + tid);
            const float x = await_value<true>(near + rs.near_stride + tid, c.seq(layer, kOproj), c);
            l.xraw[tid] = x;
            l.xs[tid] = x * gain_ffn;
        }
        lds_barrier();
    }
    u64* near_hb = c.t.near_hb + static_cast<size_t>(c.xcc) * c.t.near_hidden_stride;
    if (n_gu > 0) {
        const float scale = resident_scale(c, l.xraw);
        const float gate = row16_sum(lane_dot<kResDimLoads, kResGroup>(w_gu, l.xs, l16)) * scale;
        const float up = lane_xor(gate, 16, lane);
        if (l16 == 0 && (slot & 1) == 0 && slot < 2 * n_gu) {
            const float sigma = 1.0f / (1.0f + expf(-gate));  // ops.cpp:80-85
            publish_near(near_hb + w * rs.gu + (slot >> 1), (gate * sigma) * up, c.seq(layer, kGateUp));
        }
    }
    // x + W2 . that, to the next layer's XCD
    if (n_down > 0) {
        if (tid < hidden) l.wide[tid] = await_value<true>(near_hb + tid, c.seq(layer, kGateUp), c);
        lds_barrier();
        const float sum = wave_sum(lane_dot<kResHiddenLoads, kWave>(w_down, l.wide, lane));
        const int row = w * rs.down + wave;
        if (lane == 0 && wave < n_down) publish(c.t.x + row, l.xraw[row] + sum, c.seq(layer, kDown));
    }
    lds_barrier();
    for (int i = dim + tid; i < hidden; i += kResThreads) l.wide[i] = 0.0f;  // (zero past the next attention output again)
    lds_barrier();
}

// Nobody polls a whole vector long before it can be there: one thread looks now and then until the layer two before the
// one that forms it is done.
__device__ __forceinline__ void resident_await_turn(const Ctx& c, int layer) {
    if (layer < 1) return;
    if (threadIdx.x == 0) {
        const unsigned want = c.seq(layer - 1, kDown);
        unsigned spins = 0;
        while (static_cast<int>(tag_of(peek(c.t.x + c.rank_in_xcc % c.a.dim)) - want) < 0) {
            if (poll_give_up(c, spins)) break;
            __builtin_amdgcn_s_sleep(6);
        }
    }
    lds_barrier();
}

template <bool kGiven>
__global__ __launch_bounds__(kResThreads) void k_decode_resident(DecodeArgs a, Tagged t, Blocks b, Resident rs) {
    extern __shared__ __align__(16) float lds[];
    __shared__ Control ctl;
    __shared__ int numbered;
    const int nwg = gridDim.x, tid = static_cast<int>(threadIdx.x);
    if (tid == 0) numbered = workgroup_number(a, t, nwg);
    for (unsigned i = tid; i < sizeof(Control) / sizeof(unsigned); i += kResThreads) reinterpret_cast<unsigned*>(&ctl)[i] = 0u;
    ResidentLds l;
    l.xraw = lds;
    l.xs = l.xraw + kResDim;
    l.wide = l.xs + b.xs_floats;  // (xs runs on into the sampler's tables)
    l.qkv = l.wide + kResHidden;
    l.score = l.qkv + 3 * kResHead;
    l.part = l.score + kResPositions;
    l.cls = l.part + kResThreads / kWave * kResHead;
    for (int i = tid; i < kResDim; i += kResThreads) l.xraw[i] = l.xs[i] = 0.0f;
    for (int i = tid; i < kResHidden; i += kResThreads) l.wide[i] = 0.0f;
    __syncthreads();
    const int wg = __builtin_amdgcn_readfirstlane(numbered);
    if (wg < 0) return;
    const int token = kGiven ? t.given : min(max(__builtin_amdgcn_readfirstlane(a.step->token), 0), a.vocab - 1);
    const int n_xcc = t.n_xcc;
    Ctx c{a, t, b, ctl, t.base, nullptr, 0u, token, t.pos, t.history_len, t.temperature, t.penalty, t.r, wg, nwg, wg % n_xcc, wg / n_xcc, 0, 0};

    // This workgroup's classifier rows into LDS: requested behind its first layer's weights, and on the first layer's
    // XCD, which has no time to lose, once that layer is done.
    const int r0 = min(a.vocab, wg * b.cls), n_cls = block_rows(a.vocab, b.cls, wg), n_lds = min(n_cls, rs.cls_in_lds);
    auto request_classifier = [&]() {
        if constexpr (!kGiven) {
            const unsigned to = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)) +
                                static_cast<unsigned>((l.cls - lds) * sizeof(float));
            const char* from = a.wcls + static_cast<size_t>(r0) * a.dim * sizeof(float);
            const int bytes = n_lds * a.dim * static_cast<int>(sizeof(float));
            for (int at = 1024 * wave_index(); at < bytes; at += kResThreads / kWave * 1024)
                if (at + 16 * lane_id() < bytes) lds_request16(from + at + 16 * lane_id(), __builtin_amdgcn_readfirstlane(to + at));
        }
    };
    // (a loop to each kind of workgroup: in one, what either forms ahead of it is held in registers by both, and spills)
    const bool early = c.xcc != 0;
    bool requested = false;
    if (c.rank_in_xcc < a.n_heads) {
        for (int layer = c.xcc; layer < a.n_layers; layer += n_xcc) {
            if (early && !requested) request_classifier();
            if (!(kGiven && layer == a.n_layers - 1)) resident_attention(c, l, rs, layer, c.rank_in_xcc);
            if (!early && !requested) request_classifier();
            requested = true;
        }
    } else {
        for (int layer = c.xcc; layer < a.n_layers; layer += n_xcc) {
            resident_rows_of_layer<kGiven>(c, l, rs, layer, c.rank_in_xcc - a.n_heads, [&]() {
                if (early && !requested) request_classifier();
                resident_await_turn(c, layer - 1);
            });
            if (!early && !requested) request_classifier();
            requested = true;
        }
    }
    if constexpr (!kGiven) {
        if (!requested) request_classifier();
        const float gain = tid < a.dim ? a.rms_final[tid] : 0.0f;
        static_assert(2 * kAttScoreFloats <= kResThreads / kWave * kResHead, "the window takes the weighted values' place");
        stage_window(c, l.part, tid, kResThreads);
        resident_await_turn(c, a.n_layers - 1);
        // In two hops, as gather_values: 256 workgroups that poll the same 18 lines across the fabric get them 2.6 to 3.3 us
        // after they were published.
        const unsigned tag = c.seq(a.n_layers - 1, kDown);
        u64* near = rs.near + static_cast<size_t>(c.xcc) * 3 * rs.near_stride + 2 * rs.near_stride;
        const int share = (a.dim + nwg / n_xcc - 1) / (nwg / n_xcc), fetched = c.rank_in_xcc * share + tid;
        if (tid < share && fetched < a.dim) publish_near(near + fetched, await_value<false>(c.t.x + fetched, tag, c), tag);
        if (tid < a.dim) {
            const float x = await_value<true>(near + tid, tag, c);
            l.xraw[tid] = x;
            l.xs[tid] = x * gain;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the rows requested into LDS)
        lds_barrier();
        const float scale = resident_scale(c, l.xraw);
        const int group = lane_id() >> 4, l16 = lane_id() & 15;
        floatx4 x[kResDimLoads];
#pragma unroll
        for (int k = 0; k < kResDimLoads; ++k) x[k] = *reinterpret_cast<const floatx4*>(l.xs + 4 * (l16 + kResGroup * k));
        float* lg = l.xs + 4 * nwg;  // where sample_token has its tables in front of it
        for (int first = 0; first < n_cls; first += kResThreads / kResGroup) {
            const int row = first + 4 * wave_index() + group;
            floatx4 w[kResDimLoads];
            if (row < n_lds) {
#pragma unroll
                for (int k = 0; k < kResDimLoads; ++k) {
                    const int col = 4 * (l16 + kResGroup * k);
                    w[k] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                    if (col < a.dim) w[k] = *reinterpret_cast<const floatx4*>(l.cls + row * a.dim + col);
                }
            } else {
                request_row<kResDimLoads, kResGroup>(w, reinterpret_cast<const float*>(a.wcls) + static_cast<size_t>(r0 + row) * a.dim, l16, a.dim, row < n_cls);
            }
            const float logit = row16_sum(lane_dot(w, x)) * scale;
            if (l16 == 0 && row < n_cls) {
                lg[row] = logit;
                a.logits[r0 + row] = logit;  // raw logits stay readable after the token
            }
        }
        lds_barrier();
        if (wave_index() < kIoWaves) {
            Lds s = {};
            s.xs = l.xs;
            s.sc = l.part;
            Io io{tid, wave_index(), 0u, 0, a.step};
            sample_token(c, io, s, lg, r0, n_cls);
            if (io.it == 0 && lds_peek(&ctl.error) != 0u) report_error(a.step, 2);
        }
    }
}
