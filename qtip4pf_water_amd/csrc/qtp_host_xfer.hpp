// qtp_host_xfer.hpp -- host <-> device transfers of the reference-shaped calls:
// the caller's arrays travel as they are through pinned chunks and are turned
// into the device layout (and back) by kernels.
// Included once, in order, by qtip4pf.hip (one translation unit).
#pragma once

// The arrays of one call, packed one behind the other in ctx->xref (device, 8
// byte words), moved in chunks of XFER_CHUNK bytes through XFER_SLOTS pinned
// buffers (the host copies one chunk while the engine moves the others) and
// converted by one kernel.  Against converting on the host and one pageable,
// synchronous copy per array (and expanding the lists on the host), one update_sc
// call of 216 H2O x 32 beads:
// 4.18 ms before, 0.64 ms now (chunks of 256 KiB: 0.2 more); get_forces of 64
// H2O 206 -> 71 us.
constexpr size_t XFER_CHUNK = 1 << 20;
constexpr int XFER_SLOTS = 4;  // qtp_ctx::xev
constexpr int XFER_MAX = 8;  // arrays per call

// One array: planar [b][3][NAP] <-> [b][n_dof] (kind 0), [b][3][NMP] <->
// [b][3 n_mols] (kind 1), or 8-byte words as they are (kind 2); or 4-byte words
// of the device set to zero (kind 3, upwards only, no place in xref).
struct XferArg {
    double *dev;
    long off, words;  // place and size in xref
    int kind;
};
struct XferArgs {
    XferArg a[XFER_MAX];
    int n, n_atoms, NAP, n_mols, NMP;
};
template <bool UP>
__global__ __launch_bounds__(256) void k_xfer(XferArgs A, double *__restrict__ x)
{
    const XferArg s = A.a[blockIdx.y];
    const int per = s.kind == 0 ? A.n_atoms : A.n_mols, pitch = s.kind == 0 ? A.NAP : A.NMP;
    const long stride = (long)gridDim.x * 256, t0 = (long)blockIdx.x * 256 + threadIdx.x;
    if (s.kind == 3) {
        int *d = (int *)s.dev;
        for (long t = t0; t < s.words; t += stride) d[t] = 0;
        return;
    }
    if (s.kind == 2) {
        for (long t = t0; t < s.words; t += stride) {
            if (UP) s.dev[t] = x[s.off + t];
            else x[s.off + t] = s.dev[t];
        }
        return;
    }
    // upwards also the padding, as zeros
    const long nb = s.words / (3 * per), n = nb * 3 * (UP ? pitch : per);
    for (long t = t0; t < n; t += stride) {
        if (UP) {
            const long bd = t / pitch;
            const int i = (int)(t - bd * pitch);
            const long b = bd / 3;
            s.dev[t] = i < per ? x[s.off + b * 3 * per + 3L * i + (bd - 3 * b)] : 0.0;
        } else {
            const long bi = t / 3, b = bi / per;
            const int d = (int)(t - 3 * bi), i = (int)(bi - b * per);
            x[s.off + t] = s.dev[(b * 3 + d) * pitch + i];
        }
    }
}

static int xfer_room(qtp_ctx *ctx, size_t bytes)
{
    if (!ctx->xpin) {
        HIPCHK(hipHostMalloc((void **)&ctx->xpin, XFER_CHUNK * XFER_SLOTS, hipHostMallocDefault));
        for (int i = 0; i < XFER_SLOTS; ++i)
            HIPCHK(hipEventCreateWithFlags(&ctx->xev[i], hipEventDisableTiming));
    }
    if (bytes > ctx->xref_cap) {
        HIPCHK(hipStreamSynchronize(ctx->stream));
        if (ctx->xref) HIPCHK(hipFree(ctx->xref));
        ctx->xref = nullptr;
        ctx->xref_cap = 0;
        HIPCHK(hipMalloc((void **)&ctx->xref, bytes));
        ctx->xref_cap = bytes;
    }
    return QTP_OK;
}

// The transfer of one call: add the arrays, then up() or down().
struct Xfer {
    qtp_ctx *ctx;
    XferArgs A{};
    struct Host {
        char *p;
        size_t bytes;
    };
    std::vector<Host> host;  // in packing order; padded to 8 bytes in xref
    size_t total = 0;

    explicit Xfer(qtp_ctx *c) : ctx(c)
    {
        A.n_atoms = c->n_atoms;
        A.NAP = c->NAP;
        A.n_mols = c->n_mols;
        A.NMP = c->NMP;
    }
    // returns the array's word offset in xref
    long put(const void *h, size_t bytes)
    {
        const long off = (long)(total / 8);
        host.push_back({(char *)h, bytes});
        total += (bytes + 7) & ~(size_t)7;
        return off;
    }
    void add(double *dev, const void *h, long words, int kind)
    {
        XferArg &s = A.a[A.n++];
        s.dev = dev;
        s.off = put(h, (size_t)words * 8);
        s.words = words;
        s.kind = kind;
    }
    void planar(double *dev, const double *ref, int nb) { add(dev, ref, (long)nb * ctx->n_dof, 0); }
    void disp(double *dev, const double *ref, int nb) { add(dev, ref, (long)nb * 3 * ctx->n_mols, 1); }
    void raw(double *dev, const double *ref, long words) { add(dev, ref, words, 2); }

    void zero(int *dev, long words) { A.a[A.n++] = XferArg{(double *)dev, 0, words, 3}; }

    // f(pointer into a pinned slot, host pointer, bytes) over the pieces of
    // bytes [o, o + n) of the packed arrays
    template <class Fn>
    void pieces(size_t o, size_t n, char *slot, Fn f) const
    {
        size_t at = 0;
        for (const Host &h : host) {
            const size_t lo = std::max(at, o), hi = std::min(at + h.bytes, o + n);
            if (lo < hi) f(slot + (lo - o), h.p + (lo - at), hi - lo);
            at += (h.bytes + 7) & ~(size_t)7;
        }
    }
    dim3 grid() const
    {
        long most = 1;
        for (int i = 0; i < A.n; ++i) most = std::max(most, A.a[i].words);
        return dim3((unsigned)std::min(1024L, (most + 255) / 256), (unsigned)A.n);
    }
    // Host -> device; queued on the context's stream (the host arrays are read
    // before it returns).
    int up()
    {
        CHK(xfer_room(ctx, total));
        for (size_t o = 0; o < total; o += XFER_CHUNK) {
            const int i = ctx->xslot++ % XFER_SLOTS;
            const size_t n = std::min(XFER_CHUNK, total - o);
            char *slot = ctx->xpin + i * XFER_CHUNK;
            HIPCHK(hipEventSynchronize(ctx->xev[i]));
            pieces(o, n, slot, [](char *s, char *h, size_t b) { std::memcpy(s, h, b); });
            HIPCHK(hipMemcpyAsync((char *)ctx->xref + o, slot, n, hipMemcpyHostToDevice, ctx->stream));
            HIPCHK(hipEventRecord(ctx->xev[i], ctx->stream));
        }
        if (A.n) k_xfer<true><<<grid(), 256, 0, ctx->stream>>>(A, ctx->xref);
        HIPCHK(hipGetLastError());
        return QTP_OK;
    }
    // Device -> host; the arrays are there when it returns.
    int down()
    {
        CHK(xfer_room(ctx, total));
        k_xfer<false><<<grid(), 256, 0, ctx->stream>>>(A, ctx->xref);
        HIPCHK(hipGetLastError());
        const long nch = (long)((total + XFER_CHUNK - 1) / XFER_CHUNK);
        for (long k = 0; k < nch + XFER_SLOTS - 1; ++k) {
            // the chunk issued XFER_SLOTS - 1 turns ago, then this turn's
            const long r = k - (XFER_SLOTS - 1);
            if (r >= 0) {
                const size_t o = (size_t)r * XFER_CHUNK;
                HIPCHK(hipEventSynchronize(ctx->xev[r % XFER_SLOTS]));
                pieces(o, std::min(XFER_CHUNK, total - o), ctx->xpin + (r % XFER_SLOTS) * XFER_CHUNK,
                       [](char *s, char *h, size_t b) { std::memcpy(h, s, b); });
            }
            if (k < nch) {
                const size_t o = (size_t)k * XFER_CHUNK;
                HIPCHK(hipMemcpyAsync(ctx->xpin + (k % XFER_SLOTS) * XFER_CHUNK, (char *)ctx->xref + o,
                                      std::min(XFER_CHUNK, total - o), hipMemcpyDeviceToHost,
                                      ctx->stream));
                HIPCHK(hipEventRecord(ctx->xev[k % XFER_SLOTS], ctx->stream));
            }
        }
        return QTP_OK;
    }
};

static int upload_planar(qtp_ctx *ctx, double *dst, const double *ref, int nb)
{
    Xfer x(ctx);
    x.planar(dst, ref, nb);
    CHK(x.up());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return QTP_OK;
}

static int download_planar(qtp_ctx *ctx, const double *src, int nb, double *ref)
{
    Xfer x(ctx);
    x.planar((double *)src, ref, nb);
    return x.down();
}

// The caller's half lists of nb beads (point[b][n], entries packed from
// ent[off[b]]) into the device half and full lists: row i of the full list
// holds its partners j < i (rows that list i) ascending, then its own row.
// LE_ROWS rows a block: incoming counts of all rows (LDS atomics) and offsets,
// then a wave per row picks its incoming entries out of all entries in their
// order, which is by rising row, and looks up the rows.  All reads are
// coalesced and from L2; one block a bead with its entries in arrival order and
// sorted afterwards took 187 us for 216 x 32, this 86; 64 H2O 25, this 12.  n <=
// 1024.
// grid: nb * ceil(n / LE_ROWS), 1024 threads.
constexpr int LE_ROWS = 16;
__global__ __launch_bounds__(1024) void k_list_expand(int n, int list_size, long fcap,
                                                      const int *__restrict__ pt_in,
                                                      const int *__restrict__ ent,
                                                      const int *__restrict__ off,
                                                      int *__restrict__ point, int *__restrict__ list,
                                                      int *__restrict__ fpoint, int *__restrict__ flist)
{
    __shared__ int pt[NL_FUSED_MAXMOL], inc[NL_FUSED_MAXMOL], beg[NL_FUSED_MAXMOL];
    __shared__ int s_tot[16];
    const int nparts = (n + LE_ROWS - 1) / LE_ROWS;
    const int b = blockIdx.x / nparts, part = blockIdx.x - b * nparts;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int *H = list + (long)b * list_size, *FL = flist + (long)b * fcap;
    if (tid < n) {
        pt[tid] = pt_in[(long)b * n + tid];
        inc[tid] = 0;
    }
    __syncthreads();
    const int k0 = pt[0], k1 = pt[n - 1];
    const int *L = ent + off[b] - k0;  // entries k0 ... k1 - 1
#pragma unroll 4
    for (int k = k0 + tid; k < k1; k += 1024) {
        const int j = L[k];
        if (part == 0) H[k] = j;
        atomicAdd(&inc[j], 1);
    }
    __syncthreads();
    // offsets: thread i <-> row i (the last row of a half list is empty)
    int v = 0;
    if (tid < n) v = inc[tid] + (tid < n - 1 ? pt[tid + 1] - pt[tid] : 0);
    int s = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(s, o, 64);
        if (lane >= o) s += t;
    }
    if (lane == 63) s_tot[w] = s;
    __syncthreads();
    int base = s - v;
    for (int ww = 0; ww < w; ++ww) base += s_tot[ww];
    if (tid < n) {
        beg[tid] = base;
        if (part == 0) {
            point[(long)b * n + tid] = pt[tid];
            fpoint[(long)b * (n + 1) + tid] = base;
            if (tid == n - 1) fpoint[(long)b * (n + 1) + n] = base + v;
        }
    }
    __syncthreads();
    const int i = part * LE_ROWS + w;
    if (i >= n) return;
    const int m = inc[i], f0 = beg[i];
    const unsigned long long below = lane == 0 ? 0ull : ~0ull >> (64 - lane);
    int at = f0;
    if (m > 0) {
#pragma unroll 8
        for (int c = k0; c < k1; c += 64) {
            const int k = c + lane;
            const bool in = k < k1 && L[min(k, k1 - 1)] == i;
            const unsigned long long bal = __ballot(in);
            if (in) FL[at + __popcll(bal & below)] = k;
            at += __popcll(bal);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        for (int t = lane; t < m; t += 64) {
            // the row that holds entry k: the last one with pt <= k
            const int k = FL[f0 + t];
            int lo = 0, hi = n - 1;  // pt[lo] <= k < pt[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (pt[mid] <= k) lo = mid;
                else hi = mid;
            }
            FL[f0 + t] = lo;
        }
    }
    if (i < n - 1)
        for (int k = pt[i] + lane; k < pt[i + 1]; k += 64) FL[f0 + m + k - pt[i]] = L[k];
}

// Caller's half lists (reference layout) checked: rows rise within list_size,
// entries are molecules.  Row n_mols-1 is ignored as forces.cpp:489 does.
static int check_lists(qtp_ctx *ctx, const int *point, const int *list, int b0, int nb)
{
    const int n = ctx->n_mols;
    for (int b = b0; b < b0 + nb; ++b) {
        const int *pt = point + (long)b * n;
        const int *ls = list + (long)b * ctx->list_size;
        for (int i = 0; i < n - 1; ++i) {
            if (pt[i] < 0 || pt[i + 1] > ctx->list_size || pt[i + 1] < pt[i]) {
                ctx->err = "neighbour list: point[] out of range";
                return QTP_ERR_ARG;
            }
            bool bad = false;
            for (int k = pt[i]; k < pt[i + 1]; ++k) bad |= (unsigned)ls[k] >= (unsigned)n;
            if (bad) {
                ctx->err = "neighbour list: entry out of range";
                return QTP_ERR_ARG;
            }
        }
        if (n > 1 && 2L * (pt[n - 1] - pt[0]) > ctx->fcap) {
            ctx->err = "neighbour list: full list exceeds capacity";
            return QTP_ERR_LIST_OVERFLOW;
        }
    }
    return QTP_OK;
}

// Caller's half lists -> device half + full lists, expanded on the host (more
// molecules than k_list_expand takes).
static int upload_lists_host(qtp_ctx *ctx, const int *point, const int *list, int b0, int nb,
                             int dev_b0)
{
    const int n = ctx->n_mols;
    std::vector<int> fp((size_t)nb * (n + 1)), fl((size_t)nb * ctx->fcap, 0), cur(n);
    for (int bb = 0; bb < nb; ++bb) {
        const int *pt = point + (long)(b0 + bb) * n;
        const int *ls = list + (long)(b0 + bb) * ctx->list_size;
        int *FP = fp.data() + (size_t)bb * (n + 1), *FL = fl.data() + (size_t)bb * ctx->fcap;
        std::fill(cur.begin(), cur.end(), 0);
        for (int k = pt[0]; k < pt[n - 1]; ++k) ++cur[ls[k]];
        int pos = 0;
        for (int i = 0; i < n; ++i) {
            FP[i] = pos;
            const int m = cur[i];
            cur[i] = pos;  // partners j < i (i in row j), then row i
            pos += m + (i < n - 1 ? pt[i + 1] - pt[i] : 0);
        }
        FP[n] = pos;
        for (int i = 0; i < n - 1; ++i)
            for (int k = pt[i]; k < pt[i + 1]; ++k) FL[cur[ls[k]]++] = i;
        for (int i = 0; i < n - 1; ++i)
            for (int k = pt[i]; k < pt[i + 1]; ++k) FL[cur[i]++] = ls[k];
    }
    HIPCHK(hipMemcpy(ctx->fpoint + (size_t)dev_b0 * (n + 1), fp.data(), fp.size() * sizeof(int),
                     hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->flist + (size_t)dev_b0 * ctx->fcap, fl.data(), fl.size() * sizeof(int),
                     hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->point + (size_t)dev_b0 * n, point + (long)b0 * n, (size_t)nb * n * sizeof(int),
                     hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->list + (size_t)dev_b0 * ctx->list_size, list + (long)b0 * ctx->list_size,
                     (size_t)nb * ctx->list_size * sizeof(int), hipMemcpyHostToDevice));
    return QTP_OK;
}

// The arrays already in x and the caller's half lists (checked) of beads b0 ...
// into dev_b0 ..., in one transfer where the device expands the lists.
static int upload_with_lists(qtp_ctx *ctx, Xfer &x, const int *point, const int *list, int b0, int nb,
                             int dev_b0)
{
    const int n = ctx->n_mols;
    if (n > NL_FUSED_MAXMOL) {
        CHK(x.up());
        return upload_lists_host(ctx, point, list, b0, nb, dev_b0);
    }
    std::vector<int> off(nb);
    const long at_pt = x.put(point + (long)b0 * n, (size_t)nb * n * sizeof(int));
    const long at_off = x.put(off.data(), (size_t)nb * sizeof(int));
    long at_ent = -1;
    for (int b = 0; b < nb; ++b) {
        const int *pt = point + (long)(b0 + b) * n;
        const long at = x.put(list + (long)(b0 + b) * ctx->list_size + pt[0],
                              (size_t)(pt[n - 1] - pt[0]) * sizeof(int));
        if (b == 0) at_ent = at;
        off[b] = (int)(2 * (at - at_ent));
    }
    // nothing of an earlier list around the entries (k_list_expand itself takes
    // 98 instead of 86 us when it clears them)
    x.zero(ctx->list + (size_t)dev_b0 * ctx->list_size, (long)nb * ctx->list_size);
    CHK(x.up());
    const int *w = (const int *)ctx->xref;
    k_list_expand<<<nb * ((n + LE_ROWS - 1) / LE_ROWS), 1024, 0, ctx->stream>>>(
        n, ctx->list_size, ctx->fcap, w + 2 * at_pt, w + 2 * at_ent, w + 2 * at_off,
        ctx->point + (size_t)dev_b0 * n, ctx->list + (size_t)dev_b0 * ctx->list_size,
        ctx->fpoint + (size_t)dev_b0 * (n + 1), ctx->flist + (size_t)dev_b0 * ctx->fcap);
    HIPCHK(hipGetLastError());
    return QTP_OK;
}

// The half lists of the beads that the last step rebuilt: a bead's entries and
// zeros up to list_size, the row the list kernels write (neighbour.cpp:23-32).
// Only the entries travel.
static int download_rebuilt(qtp_ctx *ctx, int *point, int *list)
{
    const int n = ctx->n_mols;
    std::vector<int> fl(ctx->P);
    HIPCHK(hipMemcpy(fl.data(), ctx->flag, ctx->P * sizeof(int), hipMemcpyDeviceToHost));
    for (int b = 0; b < ctx->P; ++b) {
        if (!fl[b]) continue;
        int *pt = point + (long)b * n, *ls = list + (long)b * ctx->list_size;
        HIPCHK(hipMemcpy(pt, ctx->point + (size_t)b * n, n * sizeof(int), hipMemcpyDeviceToHost));
        HIPCHK(hipMemcpy(ls, ctx->list + (size_t)b * ctx->list_size, pt[n - 1] * sizeof(int),
                         hipMemcpyDeviceToHost));
        std::fill(ls + pt[n - 1], ls + ctx->list_size, 0);
    }
    return QTP_OK;
}

static int check_finite(qtp_ctx *ctx, const double *a, long n, const char *what)
{
    constexpr uint64_t EXP = 0x7ff0000000000000ull;
    uint64_t bad = 0;
    for (long i = 0; i < n; ++i) {
        uint64_t u;
        std::memcpy(&u, a + i, 8);
        bad |= (uint64_t)((u & EXP) == EXP);
    }
    if (bad) {
        ctx->err = std::string(what) + " contains a non-finite value";
        return QTP_ERR_NONFINITE;
    }
    return QTP_OK;
}
