// shell_blocks.h -- the shell analysis by shell blocks, included by shell_analyse.hip inside
// its namespace after the device helpers it shares with the lane-per-peak kernels.
//
// The crossing pass gives every peak its gather extent before any gather, and a shell's sums
// start from zero and depend on no other shell.  So the gather's unit of work here is not a
// peak but four consecutive shells of a peak (a block): peaks of 170 and of 14 000 cells give
// work items of similar length, a wavefront's 64 lanes take blocks of the same shells, and
// the items of a single deep peak run side by side (one lane per peak ran as long as its
// wavefront's deepest peak: 5.7 of the 7.4 ms of a 128^3 tile).  Within a shell the cells are
// summed in the reference's order by one lane, with the reference's Float32 products, so the
// profile is the lane-per-peak kernels' bit for bit.  The fields are read as the caller gave
// them: no cell records are written.
//
// Measured against the lane-per-peak kernel with its records (same bits): shell analysis of the
// 1024^3 tile 327 -> 211 ms, of the 512^3 tile 51.6 -> 25.8 ms, of a 128^3 tile 7.9 -> 1.10 ms, of a
// 40^3 tile 1.33 -> 0.37 ms, of 24 tiles of 96^3 to 256^3 in one call 37.6 -> 20.9 ms.  Calls that a
// lane per peak answers quicker stay with that kernel (analyse_tiles, lanes_quicker).
//
// A block's sums are five 128-byte lines side by side, one per field (delta, its transpose,
// psi_1 xyz), four doubles per shell: {F, G0, G1, G2}, {H0, H1, H2, -}, {S, R0, R1, R2} x 3;
// G, H and R divided by the shell's radius.  Shell s of a peak is in its block s / 4 (the
// first block's shell 0 is unused).  What reads them takes four lanes per peak, a shell each: a
// line is one peak's four lanes' 128 bytes, fetched once.

constexpr int BLK = 4;          // shells per block
constexpr int BLK_FIELDS = 5;   // lines per block
constexpr int BLK_LINES = BLK_FIELDS * 4 * BLK;  // doubles of a block's lines
constexpr int BLK_DOUBLES = BLK_LINES + BLK;     // ... and Fbar of its 4 shells

struct BlockArgs {
    const int32_t* stop;   // per global peak id: last shell of the gather
    int32_t* cross;        // per global peak id: crossing shell, 0 = none; then, from the radial
                           // logic on, the first shell beyond RTHL's, 0 = no collapse
    const int64_t* base;   // per global peak id: first block of its profile
    int64_t e0, ne;        // blocks [e0, e0 + ne) are the ones of this launch
    double* prof;          // [BLK_LINES ne] the blocks' lines
    double* fb;            // [4 ne] Fbar of each shell
    const uint32_t* cell8; // offsets of every table cell: three signed bytes
    const double* rinv;    // 1 / rad of each shell
    const int32_t* win;    // per shell s: last m1 with rad < rad[s] + 2, last with <=, first
                           // with rad > rad[s] - 2 (not below 0)
};

// Shell s of the profile that starts at block eb: its doubles of field f are at 4 BLK f.
__device__ __forceinline__ double* entry_of(const BlockArgs& B, int64_t eb, int s) {
    return B.prof + (eb + (s >> 2)) * BLK_LINES + (s & 3) * 4;
}

__device__ __forceinline__ int blocks_of(int stop) { return (stop >> 2) + 1; }

__global__ void block_count_kernel(const int32_t* __restrict__ vals,
                                   const int32_t* __restrict__ stop, int64_t ntot,
                                   int32_t* __restrict__ cnt) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < ntot) cnt[q] = blocks_of(stop[vals ? vals[q] : q]);
}

__global__ void block_base_kernel(const int32_t* __restrict__ vals,
                                  const int64_t* __restrict__ off, int64_t ntot,
                                  int64_t* __restrict__ base) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < ntot) base[vals ? vals[q] : q] = off[q];
}

// index of the r-th set bit of m (r < popcount)
__device__ __forceinline__ int nth_bit(uint64_t m, int r) {
    int pos = 0;
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
        const uint64_t low = m & ((1ull << w) - 1ull);
        const int c = __popcll(low);
        const bool up = r >= c;
        r -= up ? c : 0;
        pos += up ? w : 0;
        m = up ? m >> w : low;
    }
    return pos;
}

__device__ __forceinline__ int byte_of(uint32_t w, int q) {
    return (int)(int8_t)((w >> (8 * q)) & 0xffu);
}

// a / r, correctly rounded, with y = 1 / r correctly rounded: two Newton steps on the quotient
// (the second, from a quotient already within an ulp, rounds it correctly: Markstein, IBM J.
// Res. Dev. 34, 1990), 5 operations instead of the division's 12.  An infinite or NaN a keeps
// its product.  Checked against the division in tests/test_shell_blocks_cpu.py.
__device__ __forceinline__ double div_rad(double a, double r, double y) {
    const double q0 = a * y;
    const double q1 = fma(fma(-q0, r, a), y, q0);
    const double q2 = fma(fma(-q1, r, a), y, q1);
    return fabs(q0) <= 1.7976931348623157e308 ? q2 : q0;
}

// The peak's ball of radius R (cells) leaves the grid.
__device__ __forceinline__ bool ball_outside(const TileDev& T, int ci, int cj, int ck, int R) {
    return !(ci - R >= 1 && ci + R <= T.n && cj - R >= 1 && cj + R <= T.n && ck - R >= 1 &&
             ck + R <= T.n);
}

// ------------------------------------------------------------------ gather from bricks
// The blocks within BR_H cells (97 % of the 1024^3 tile's peaks entirely, 90 % of its cells):
// a workgroup takes the peaks of one 16^3 brick of the first order and stages the brick with
// an 8-cell halo, 32^3 floats of one field at a time, in LDS (128 KB of the CU's 160), each
// wavefront load bringing whole rows; the items of the brick then sum their shells from LDS.
// An item is a lane's; its offsets come from a table in LDS, so that a wavefront may mix
// blocks (a brick has some 120 peaks, few of them deep).  One field needs 4 FP64 sums, so the
// five fields take turns in the one box: with all eight values of a cell side by side the box
// would hold a brick of 17 cells halo included.
constexpr int BR_CORE = 16, BR_H = 8, BR_W = 32, BR_T = 1024;
constexpr int BR_PK = 256;      // peaks at a time, at most
constexpr int BR_SH = 64;       // shells within BR_H, at most
constexpr int BR_CELLS = 2112;  // cells within BR_H (2109), padded
constexpr int BR_ITEMS = 4864;  // items at a time (a brick of the 1024^3 tile has some 2900)

struct BrickArgs {
    const int64_t* start;   // [count + 1] sorted position of each brick's first peak
    const int32_t* tile;    // [count]
    const int32_t* count;
    const int32_t* vals;    // global peak id by sorted position
    const uint2* tab;       // [2][ncell]: box offset (16 bits) and offsets as Float16; then the
                            // transposed field's
    const uint8_t* order;   // [nsh] shells within BR_H by falling number of cells
    int ncell, nsh;         // cells and shells within BR_H
};

// v times the Float16 in the low or high half of w, as a Float32 product: an FMA with mz = -0,
// which leaves every product as it is (-0 and NaN included), in the form that takes the half as it
// is (a conversion and a multiply otherwise: 3 of the 18 operations of a cell)
template <bool HIGH>
__device__ __forceinline__ float mul_half(float v, uint32_t w, float mz) {
    float r;
    if (HIGH)
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(v), "v"(w), "s"(mz));
    else
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(v), "v"(w), "s"(mz));
    return r;
}

// The box value at byte address `cen` + 4 (the signed 16-bit offset in the low half of w)
__device__ __forceinline__ float box_at(uint32_t cen, uint32_t w) {
    uint32_t at;
    asm("v_mad_i32_i16 %0, %1, 4, %2" : "=v"(at) : "v"(w), "v"(cen));
    return *(const __attribute__((address_space(3))) float*)at;
}

struct BrickLds {
    float box[BR_W * BR_W * BR_W];
    uint2 tab[BR_CELLS];
    uint64_t mask[BR_SH * (BR_PK / 64)];
    double rad[BR_SH], rinv[BR_SH];
    int base[BR_PK];
    int ctr[BLK_FIELDS], np, tot;
    uint16_t cen[BR_PK], cenT[BR_PK];
    uint16_t pre[BR_SH * (BR_PK / 64)];
    uint16_t sstart[BR_SH + 1];
    uint16_t item[BR_ITEMS];  // shell << 8 | peak, shells of most cells first
    uint8_t stop[BR_PK];
};
static_assert(sizeof(BrickLds) <= 160 * 1024, "one brick per CU");

template <bool VEC4>
__device__ __forceinline__ void stage_box(float* box, const float* __restrict__ f, int n, int f0,
                                          int r0, int q0, int64_t s1, int64_t s2) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // cells outside the grid are read as its nearest cell: no item that needs them is here
    if (VEC4) {
        const int fx = min(max(f0 + 4 * (lane & 7), 0), n - 4);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int g = k * (BR_T / 64) + wave, row = g * 8 + (lane >> 3);
            const int r = min(max(r0 + (row & 31), 0), n - 1), q = min(max(q0 + (row >> 5), 0), n - 1);
            __builtin_amdgcn_global_load_lds(
                f + fx + r * s1 + q * s2,
                (__attribute__((address_space(3))) void*)(box + g * 256), 16, 0, 0);
        }
    } else {
        const int fx = min(max(f0 + (lane & 31), 0), n - 1);
#pragma unroll 8
        for (int k = 0; k < 32; ++k) {
            const int g = k * (BR_T / 64) + wave, row = g * 2 + (lane >> 5);
            const int r = min(max(r0 + (row & 31), 0), n - 1), q = min(max(q0 + (row >> 5), 0), n - 1);
            __builtin_amdgcn_global_load_lds(
                f + fx + r * s1 + q * s2,
                (__attribute__((address_space(3))) void*)(box + g * 64), 4, 0, 0);
        }
    }
}

__device__ __forceinline__ void store4(double* __restrict__ p, double a, double b, double c,
                                       double d) {
    reinterpret_cast<double2*>(p)[0] = make_double2(a, b);
    reinterpret_cast<double2*>(p)[1] = make_double2(c, d);
}

// The items of one field: sums of v, v dx, v dy, v dz (PLAIN: the first too) of every item's
// shell.  A wavefront takes 64 items at a time.
template <bool PLAIN>
__device__ __forceinline__ void brick_items(BrickLds& L, int tot, int* ctr,
                                            const uint16_t* __restrict__ cen,
                                            double* __restrict__ line) {
    const int lane = threadIdx.x & 63;
    for (;;) {
        int t0 = 0;
        if (lane == 0) t0 = atomicAdd(ctr, 64);
        t0 = __builtin_amdgcn_readfirstlane(t0);
        if (t0 >= tot) break;
        const int t = t0 + lane;
        if (t >= tot) continue;
        const int it = L.item[t], q = it & 255, s = it >> 8;
        // LDS byte address of the peak's cell in the box
        const uint32_t c0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)L.box + 4u * cen[q];
        double* out = line + ((int64_t)L.base[q] + (s >> 2)) * BLK_LINES + (s & 3) * 4;
        double A = 0.0, A0 = 0.0, A1 = 0.0, A2 = 0.0;
        if (s == 1) {
            if (PLAIN) A = (double)box_at(c0, 0);
        } else {
            int c = L.sstart[s];
            const int e = L.sstart[s + 1];
            auto add = [&](float v, uint2 w) {
                if (PLAIN) A += (double)v;
                A0 += (double)mul_half<true>(v, w.x, -0.0f);
                A1 += (double)mul_half<false>(v, w.y, -0.0f);
                A2 += (double)mul_half<true>(v, w.y, -0.0f);
            };
            for (; c + 4 <= e; c += 4) {
                uint2 w[4];
                float v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) w[k] = L.tab[c + k];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = box_at(c0, w[k].x);
#pragma unroll
                for (int k = 0; k < 4; ++k) add(v[k], w[k]);
            }
            if (c < e) {  // a shell's cells come in pairs
                const uint2 w0 = L.tab[c], w1 = L.tab[c + 1];
                const float v0 = box_at(c0, w0.x), v1 = box_at(c0, w1.x);
                add(v0, w0);
                add(v1, w1);
            }
            const double r = L.rad[s], y = L.rinv[s];
            A0 = div_rad(A0, r, y);
            A1 = div_rad(A1, r, y);
            A2 = div_rad(A2, r, y);
        }
        if (PLAIN) store4(out, A, A0, A1, A2);
        else store4(out, A0, A1, A2, 0.0);
    }
}

template <bool VEC4>
__global__ __launch_bounds__(BR_T) void gather_bricks_kernel(SAArgs a, BlockArgs B, BrickArgs K) {
    extern __shared__ char lds_raw[];
    BrickLds& L = *reinterpret_cast<BrickLds*>(lds_raw);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // runs of 64 bricks (a 64^3 brick) per XCD in turn
    const int j = (int)(blockIdx.x >> 3);
    const int k = (((j >> 6) << 3) + (int)(blockIdx.x & 7)) * 64 + (j & 63);
    if (k >= *K.count) return;
    const int64_t q0 = K.start[k], q1 = K.start[k + 1];
    const TileDev& T = a.tiles[K.tile[k]];
    {
        // a brick lies in one chunk
        const int64_t e = B.base[K.vals[q0]] - B.e0;
        if (e < 0 || e >= B.ne) return;
    }
    const int p0 = (int)(K.vals[q0] - T.base);
    const int ox = ((T.pi[p0] - 1) & ~(BR_CORE - 1)) - BR_H, oy = ((T.pj[p0] - 1) & ~(BR_CORE - 1)) - BR_H,
              oz = ((T.pk[p0] - 1) & ~(BR_CORE - 1)) - BR_H;
    const int nsh = K.nsh;  // shells 1 .. nsh
    constexpr int NW = BR_PK / 64;
    // lane i's: the i-th shell by falling number of cells (read one by one as they are wanted, each
    // was a trip to the cache in a chain of 55)
    const int order = lane < nsh ? (int)K.order[lane] : 0;
    for (int s = tid; s <= nsh + 1; s += BR_T) {
        // table start of shell s, s = nsh + 1 the end of the last one
        L.sstart[s] = (uint16_t)(s < 1 ? 0 : s <= nsh ? a.shell_start[s - 1] : K.ncell);
        if (s >= 1 && s <= nsh) {
            L.rad[s] = a.rad[s];
            L.rinv[s] = B.rinv[s];
        }
    }
    int np = 0;
    for (int64_t qs = q0; qs < q1; qs += np) {
        const int npm = (int)min((int64_t)BR_PK, q1 - qs);
        int stop = 0;  // shells of this thread's peak, 0: none here
        if (tid < npm) {
            const int64_t id = K.vals[qs + tid];
            const int p = (int)(id - T.base);
            const int ci = T.pi[p], cj = T.pj[p], ck = T.pk[p];
            const int st = B.stop[id];
            if (!ball_outside(T, ci, cj, ck, min(BR_H, (int)a.rad[st]))) stop = min(st, nsh);
            const int x = ci - 1 - ox, y = cj - 1 - oy, z = ck - 1 - oz;
            L.base[tid] = (int)(B.base[id] - B.e0);
            L.cen[tid] = (uint16_t)(x + BR_W * y + BR_W * BR_W * z);
            L.cenT[tid] = (uint16_t)(z + BR_W * x + BR_W * BR_W * y);
            L.stop[tid] = (uint8_t)stop;
        }
        __syncthreads();
        // as many peaks as the item list holds
        if (wave == 0) {
            int n = 0, sum = 0;
            for (int w = 0; w < NW; ++w) {
                const int i = w * 64 + lane;
                int run = i < npm ? (int)L.stop[i] : 0;
                for (int d = 1; d < 64; d <<= 1) {
                    const int o = __shfl_up(run, d);
                    if (lane >= d) run += o;
                }
                n += (int)__popcll(__ballot(i < npm && sum + run <= BR_ITEMS));
                sum += __shfl(run, 63);
            }
            if (lane == 0) L.np = n;
            if (lane < BLK_FIELDS) L.ctr[lane] = 0;
        }
        __syncthreads();
        np = L.np;
        if (wave < NW)
            for (int i = 0; i < nsh; ++i) {
                const uint64_t m = __ballot(tid < np && stop >= __builtin_amdgcn_readlane(order, i));
                if (lane == 0) L.mask[i * NW + wave] = m;
            }
        __syncthreads();
        if (wave == 0) {
            int mine[NW], all = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                mine[w] = lane < nsh ? __popcll(L.mask[lane * NW + w]) : 0;
                all += mine[w];
            }
            int sum = all;
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(sum, d);
                if (lane >= d) sum += o;
            }
            int at = sum - all;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (lane < nsh) L.pre[lane * NW + w] = (uint16_t)at;
                at += mine[w];
            }
            if (lane == 63) L.tot = sum;
        }
        __syncthreads();
        for (int e = wave; e < nsh * NW; e += BR_T / 64) {
            const uint64_t m = L.mask[e];
            if ((m >> lane) & 1ull) {
                const int r = __popcll(m & ((1ull << lane) - 1ull));
                L.item[L.pre[e] + r] = (uint16_t)((__builtin_amdgcn_readlane(order, e / NW) << 8) | ((e & (NW - 1)) * 64 + lane));
            }
        }
        const int tot = L.tot;
        // the transposed delta first, then delta, psi_1 xyz through the other table
        const float* const src[BLK_FIELDS] = {T.delta, T.delta, T.etax, T.etay, T.etaz};
        // (all of them, or the one of workgroup y)
        const int f0 = gridDim.y > 1 ? (int)blockIdx.y : 0, f1 = gridDim.y > 1 ? f0 + 1 : BLK_FIELDS;
        for (int f = f0; f < f1 && tot > 0; ++f) {
            if (f < 2 || f == f0)
                for (int c = tid; c < K.ncell; c += BR_T) L.tab[c] = K.tab[(f == 0 ? K.ncell : 0) + c];
            if (f == 0) stage_box<VEC4>(L.box, src[f], T.n, oz, ox, oy, T.s1, T.s2);
            else stage_box<VEC4>(L.box, src[f], T.n, ox, oy, oz, T.s1, T.s2);
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (f == 0) brick_items<false>(L, tot, &L.ctr[0], L.cenT, B.prof + 4 * BLK);
            else brick_items<true>(L, tot, &L.ctr[f], L.cen, B.prof + 4 * BLK * (f == 1 ? 0 : f));
            __syncthreads();
        }
        __syncthreads();
    }
}

// Bricks of the first order: flags, then (after a scan of the flags) start and tile of each.
__global__ void brick_head_kernel(const uint64_t* __restrict__ keys, int64_t ntot, int shift,
                                  int32_t* __restrict__ flag) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < ntot) flag[q] = q == 0 || (keys[q] >> shift) != (keys[q - 1] >> shift);
}

__global__ void brick_list_kernel(const uint64_t* __restrict__ keys,
                                  const int32_t* __restrict__ flag,
                                  const int64_t* __restrict__ rank, int64_t ntot,
                                  int64_t* __restrict__ start, int32_t* __restrict__ tile,
                                  int32_t* __restrict__ count) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ntot) return;
    if (flag[q]) {
        start[rank[q]] = q;
        tile[rank[q]] = (int32_t)(keys[q] >> 50);
    }
    if (q == ntot - 1) {
        start[rank[q] + flag[q]] = ntot;
        *count = (int32_t)(rank[q] + flag[q]);
    }
}

// Peaks the bricks do not gather entirely: those whose ball leaves the grid are appended to
// their tile's slots of `slot` (all -1 before; cnt[1 + t] of them), for gather_blocks_kernel;
// those that reach beyond BR_H to `far` (cnt[0] of them), tile << 32 | peak.
__global__ void far_list_kernel(const TileDev* __restrict__ tiles, const uint64_t* __restrict__ keys,
                                const int32_t* __restrict__ vals, const int32_t* __restrict__ stop,
                                const double* __restrict__ rad, int64_t ntot, int nsh,
                                const int64_t* __restrict__ tile_pad, int32_t* __restrict__ cnt,
                                int32_t* __restrict__ slot, int64_t* __restrict__ far) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool deep = false;
    int t = 0, p = 0;
    if (q < ntot) {
        t = (int)(keys[q] >> 50);
        const TileDev& T = tiles[t];
        const int64_t id = vals[q];
        p = (int)(id - T.base);
        const int s = stop[id];
        if (ball_outside(T, T.pi[p], T.pj[p], T.pk[p], (int)rad[s]))
            slot[tile_pad[t] + atomicAdd(&cnt[1 + t], 1)] = p;
        else deep = s > nsh;
    }
    const int lane = threadIdx.x & 63;
    const uint64_t m = __ballot(deep);
    if (m == 0) return;
    int at = 0;
    if (lane == 0) at = atomicAdd(&cnt[0], (int)__popcll(m));
    at = __builtin_amdgcn_readfirstlane(at) + (int)__popcll(m & ((1ull << lane) - 1ull));
    if (deep) far[at] = ((int64_t)t << 32) | (int64_t)p;
}

// The shells beyond BR_H of the deep peaks, one field per launch: a wavefront per peak, a lane
// per shell, read from the field as it is.  A peak's ball is read many times over (every lane
// its own cells), its neighbours' balls overlap it (the list is in brick order), and a launch
// of one field keeps what an XCD's resident peaks read within its L2; with the fields in turn,
// or each peak's box brought into LDS first, four of five lines came from beyond it.
// The transposed delta (f = 1) enters a record only through kernel_strain at the collapse, so its
// launch follows the walk and takes the collapsed peaks' shells within reach of that (1024^3
// tile, the five launches: 60 -> 45 ms).
constexpr int FAR_T = 256, FAR_WG = 4;  // workgroups per CU

__global__ __launch_bounds__(FAR_T) void gather_far_kernel(SAArgs a, BlockArgs B,
                                                           const int64_t* __restrict__ far,
                                                           const int32_t* __restrict__ count,
                                                           int nsh, int f0) {
    // one field, or (f0 < 0) delta and psi_1 by workgroup y
    const int f = f0 >= 0 ? f0 : blockIdx.y == 0 ? 0 : (int)blockIdx.y + 1;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    constexpr int NWV = FAR_T / 64;
    const int nfar = *count, G = (int)(gridDim.x >> 3) * NWV;
    const bool tr = f == 1;  // the transposed delta
    // runs of 64 peaks per XCD in turn
    for (int l = (int)(blockIdx.x >> 3) * NWV + wave;; l += G) {
        const int i = (((l >> 6) << 3) + (int)(blockIdx.x & 7)) * 64 + (l & 63);
        if ((l >> 6) * 512 >= nfar) break;
        if (i >= nfar) continue;
        const int64_t e = far[i];
        const TileDev& T = a.tiles[__builtin_amdgcn_readfirstlane((int)(e >> 32))];
        const int p = __builtin_amdgcn_readfirstlane((int)(e & 0xffffffff));
        const int64_t eb = B.base[T.base + p] - B.e0;
        if (eb < 0 || eb >= B.ne) continue;
        int stop = B.stop[T.base + p];
        if (tr) {  // after the walk: only what kernel_strain at the collapse reads
            const int mc = B.cross[T.base + p];
            if (mc <= 0) continue;
            stop = min(stop, B.win[3 * mc + 1]);
        }
        const int s1 = T.n, s2 = T.n * T.n;
        const int ci = T.pi[p] - 1, cj = T.pj[p] - 1, ck = T.pk[p] - 1;
        const float* __restrict__ src = f <= 1 ? T.delta : f == 2 ? T.etax : f == 3 ? T.etay : T.etaz;
        // strides of i, j and k in the field read
        const int ax = tr ? s1 : 1, ay = tr ? s2 : s1, az = tr ? 1 : s2;
        src += (int64_t)ci * ax + (int64_t)cj * ay + (int64_t)ck * az;
        for (int s = nsh + 1 + lane; s <= stop; s += 64) {
            int c = a.shell_start[s - 1];
            const int en = c + a.shell_count[s - 1];
            double A = 0.0, A0 = 0.0, A1 = 0.0, A2 = 0.0;
            auto at = [&](uint32_t w) {
                return src[byte_of(w, 0) * ax + byte_of(w, 1) * ay + byte_of(w, 2) * az];
            };
            auto add = [&](float v, uint32_t w) {
                A += (double)v;
                A0 += (double)(v * (float)byte_of(w, 0));
                A1 += (double)(v * (float)byte_of(w, 1));
                A2 += (double)(v * (float)byte_of(w, 2));
            };
            for (; c + 8 <= en; c += 8) {
                uint32_t w[8];
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) w[u] = B.cell8[c + u];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = at(w[u]);
#pragma unroll
                for (int u = 0; u < 8; ++u) add(v[u], w[u]);
            }
            if (c < en) {  // up to seven more, loaded together
                uint32_t w[7];
                float v[7];
#pragma unroll
                for (int u = 0; u < 7; ++u) w[u] = B.cell8[min(c + u, en - 1)];
#pragma unroll
                for (int u = 0; u < 7; ++u) v[u] = at(w[u]);
#pragma unroll
                for (int u = 0; u < 7; ++u)
                    if (c + u < en) add(v[u], w[u]);
            }
            const double r = a.rad[s], y = B.rinv[s];
            A0 = div_rad(A0, r, y);
            A1 = div_rad(A1, r, y);
            A2 = div_rad(A2, r, y);
            double* o = entry_of(B, eb, s) + 4 * BLK * f;
            if (tr) store4(o, A0, A1, A2, 0.0);
            else store4(o, A, A0, A1, A2);
        }
    }
}

// ------------------------------------------------------------------ gather from the fields
// The peaks whose balls leave the grid (far_list_kernel's slots), read from the fields as they are.
struct BlockSums {
    double F, G0, G1, G2, H0, H1, H2;
    double S0, S1, S2, R00, R01, R02, R10, R11, R12, R20, R21, R22;
    __device__ __forceinline__ void zero() {
        F = G0 = G1 = G2 = H0 = H1 = H2 = 0.0;
        S0 = S1 = S2 = R00 = R01 = R02 = R10 = R11 = R12 = R20 = R21 = R22 = 0.0;
    }
    // the reference's Float32 products, added in FP64
    __device__ __forceinline__ void add(float d, float t, float x, float y, float z, float fx,
                                        float fy, float fz) {
        F += (double)d;
        G0 += (double)(d * fx);
        G1 += (double)(d * fy);
        G2 += (double)(d * fz);
        H0 += (double)(t * fx);
        H1 += (double)(t * fy);
        H2 += (double)(t * fz);
        S0 += (double)x;
        R00 += (double)(x * fx);
        R01 += (double)(x * fy);
        R02 += (double)(x * fz);
        S1 += (double)y;
        R10 += (double)(y * fx);
        R11 += (double)(y * fy);
        R12 += (double)(y * fz);
        S2 += (double)z;
        R20 += (double)(z * fx);
        R21 += (double)(z * fy);
        R22 += (double)(z * fz);
    }
};


struct BlockFields {
    const float *d, *x, *y, *z;
};

// The shell's sums of one lane: cells [st, st + nc) of the table around the peak whose cell is
// c0 (cT in the transposed field); cells outside the grid are skipped.
__device__ __forceinline__ void block_shell(const BlockFields& f, const uint32_t* __restrict__ cell8,
                                            int st, int nc, int n, int ci, int cj, int ck,
                                            int64_t c0, int64_t cT, BlockSums& A) {
    const int s1 = n, s2 = n * n;
    for (int c = 0; c < nc; ++c) {
        const uint32_t w = cell8[st + c];
        const int ox = byte_of(w, 0), oy = byte_of(w, 1), oz = byte_of(w, 2);
        const int i1 = ci + ox, i2 = cj + oy, i3 = ck + oz;
        if (i1 < 1 || i1 > n || i2 < 1 || i2 > n || i3 < 1 || i3 > n) continue;
        const int64_t o = c0 + (ox + oy * s1 + oz * s2);
        A.add(f.d[o], f.d[cT + (oz + ox * s1 + oy * s2)], f.x[o], f.y[o], f.z[o], (float)ox,
              (float)oy, (float)oz);
    }
}

// Gather of the blocks of 64 schedule slots (a workgroup per group and share of its items):
// the first wavefront lists, for each block index b, which of the group's peaks reach it; item
// t is the (t - first item of b)-th of them.
__global__ __launch_bounds__(256) void gather_blocks_kernel(SAArgs a, BlockArgs B, int64_t g0,
                                                            int64_t ng, int shares) {
    extern __shared__ uint64_t lds[];
    const int nbmax = (a.NS >> 2) + 1;
    uint64_t* mask = lds;                    // [nbmax] peaks with more than b blocks
    int* pre = (int*)(mask + nbmax);         // [nbmax + 1] items before block b
    __shared__ int64_t s_base[64];
    __shared__ int s_pos[3][64], s_stop[64], s_nb;
    // contiguous runs of groups per XCD (workgroups are dealt to the XCDs in turn)
    const int64_t nwg = (int64_t)gridDim.x, per = nwg >> 3;
    const int64_t w = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int64_t g = g0 + w / shares;
    const int share = (int)(w % shares);
    if (g >= g0 + ng) return;
    const TileDev& T = a.tiles[a.gtile[g]];
    const int tid = threadIdx.x;
    if (tid < 64) {
        const int p = a.slot[g * 64 + tid];
        int nb = 0;
        if (p >= 0) {
            const int64_t b0 = B.base[T.base + p] - B.e0;
            if (b0 >= 0 && b0 < B.ne) {
                const int stop = B.stop[T.base + p];
                nb = blocks_of(stop);
                s_base[tid] = b0;
                s_stop[tid] = stop;
                s_pos[0][tid] = T.pi[p];
                s_pos[1][tid] = T.pj[p];
                s_pos[2][tid] = T.pk[p];
            }
        }
        int sum = 0, b = 0;
        for (; b < nbmax; ++b) {
            const uint64_t m = __ballot(nb > b);
            if (m == 0) break;
            if (tid == 0) {
                mask[b] = m;
                pre[b] = sum;
            }
            sum += __popcll(m);
        }
        if (tid == 0) {
            pre[b] = sum;
            s_nb = b;
        }
    }
    __syncthreads();
    const int nb = s_nb, tot = pre[nb];
    const BlockFields f{T.delta, T.etax, T.etay, T.etaz};
    for (int t0 = share * 256 + (tid & ~63); t0 < tot; t0 += 256 * shares) {
        const int t = t0 + (tid & 63);
        const bool on = t < tot;
        int lo = 0, hi = nb - 1;  // last b with pre[b] <= t
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (pre[mid] <= t) lo = mid;
            else hi = mid - 1;
        }
        const int b = lo;
        const int q = on ? nth_bit(mask[b], t - pre[b]) : 0;
        const int stop = on ? s_stop[q] : 0;
        const int ci = s_pos[0][q], cj = s_pos[1][q], ck = s_pos[2][q];
        const int n = T.n;
        const int64_t c0 = (int64_t)(ci - 1) + (cj - 1) * T.s1 + (ck - 1) * T.s2;
        const int64_t cT = (int64_t)(ck - 1) + (ci - 1) * T.s1 + (cj - 1) * T.s2;
        const int64_t e = on ? s_base[q] + b : 0;
        for (int u = 0; u < BLK; ++u) {
            const int s = BLK * b + u;
            if (s < 1 || s > stop) continue;
            BlockSums A;
            A.zero();
            if (s == 1) {
                // the peak's cell: its values and no first-order terms
                A.F = (double)f.d[c0];
                A.S0 = 0.0 + (double)f.x[c0];
                A.S1 = 0.0 + (double)f.y[c0];
                A.S2 = 0.0 + (double)f.z[c0];
            } else {
                const int st = a.shell_start[s - 1], nc = a.shell_count[s - 1];
                block_shell(f, B.cell8, st, nc, n, ci, cj, ck, c0, cT, A);
                const double r = a.rad[s], y = B.rinv[s];
                for (double* v : {&A.G0, &A.G1, &A.G2, &A.H0, &A.H1, &A.H2, &A.R00, &A.R01, &A.R02,
                                  &A.R10, &A.R11, &A.R12, &A.R20, &A.R21, &A.R22})
                    *v = div_rad(*v, r, y);
            }
            double* o = B.prof + e * BLK_LINES + u * 4;
            store4(o, A.F, A.G0, A.G1, A.G2);
            store4(o + 16, A.H0, A.H1, A.H2, 0.0);
            store4(o + 32, A.S0, A.R00, A.R01, A.R02);
            store4(o + 48, A.S1, A.R10, A.R11, A.R12);
            store4(o + 64, A.S2, A.R20, A.R21, A.R22);
        }
    }
}

// Cells of shell s inside the grid around a peak (all of them unless the ball leaves it).
__device__ __forceinline__ int shell_cells_in(const SAArgs& a, const TileDev& T, int s, int ci,
                                              int cj, int ck, bool out) {
    const int nc = a.shell_count[s - 1];
    if (!out) return nc;
    const int st = a.shell_start[s - 1];
    int in = 0;
    for (int c = 0; c < nc; ++c) {
        const int4 o = a.cells[st + c];
        const int i1 = ci + o.x, i2 = cj + o.y, i3 = ck + o.z;
        in += i1 >= 1 && i1 <= T.n && i2 >= 1 && i2 <= T.n && i3 >= 1 && i3 <= T.n;
    }
    return in;
}

// Fbar of every gathered shell (RadialShell.jl:410-416), a lane per peak of slots
// [s0, s0 + ns): a serial recurrence over the shells' delta sums.
__global__ __launch_bounds__(64) void block_fbar_kernel(SAArgs a, BlockArgs B, int64_t g0) {
    const int64_t g = g0 + blockIdx.x;
    const TileDev& T = a.tiles[a.gtile[g]];
    const int p = a.slot[g * 64 + threadIdx.x];
    if (p < 0) return;
    const int64_t eb = B.base[T.base + p] - B.e0;
    if (eb < 0 || eb >= B.ne) return;
    const int stop = B.stop[T.base + p];
    const int ci = T.pi[p], cj = T.pj[p], ck = T.pk[p];
    const bool out = ball_outside(T, ci, cj, ck, (int)a.rad[stop]);
    const double* L = B.prof + eb * BLK_LINES;
    double* fb = B.fb + eb * BLK;
    // the four sums of a block's line together, the next line's on their way meanwhile (shell by
    // shell, with 32 wavefronts per CU, every sum fetched its line anew)
    double Fprev = L[4], dFbarp = Fprev, Fn[BLK];
#pragma unroll
    for (int u = 0; u < BLK; ++u) Fn[u] = L[u * 4];
    for (int s0 = 0; s0 <= stop; s0 += BLK) {
        double F[BLK], Fb[BLK];
#pragma unroll
        for (int u = 0; u < BLK; ++u) F[u] = Fn[u];
        if (s0 + BLK <= stop) {
#pragma unroll
            for (int u = 0; u < BLK; ++u) Fn[u] = L[(s0 / BLK + 1) * BLK_LINES + u * 4];
        }
#pragma unroll
        for (int u = 0; u < BLK; ++u) {
            const int s = s0 + u;
            if (s >= 2 && s <= stop) {
                const int nin = shell_cells_in(a, T, s, ci, cj, ck, out);
                const double dFbar = nin > 0 ? F[u] / (double)nin : 0.0;
                const double rad3p = cube(a.rad[s - 1]), rad3 = cube(a.rad[s]);
                Fprev = (rad3p * Fprev + 0.5 * (dFbarp + dFbar) * (rad3 - rad3p)) / rad3;
                dFbarp = dFbar;
            }
            Fb[u] = Fprev;
        }
        store4(fb + s0, Fb[0], Fb[1], Fb[2], Fb[3]);
    }
}

// Rows of a launch: slots [slot0, slot0 + nslot), NR = 64 / W per wavefront, contiguous runs per
// XCD.  False: this wavefront has no slot.
template <int W>
__device__ __forceinline__ bool row_slot(int64_t nslot, int64_t& first) {
    constexpr int NR = 64 / W;
    const int64_t per = (int64_t)gridDim.x >> 3;
    first = ((int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3)) * NR;
    return first < nslot;
}

// block_fbar_kernel for few peaks, where its time is the deepest peak's chain of loads: sixteen
// lanes per peak, a shell each; the recurrence then runs over their quotients in order, every lane
// alike.  128^3 tile 67 -> 50 us.
__global__ __launch_bounds__(64) void fbar_rows_kernel(SAArgs a, BlockArgs B, int64_t slot0,
                                                       int64_t nslot) {
    constexpr int W = 16;
    const int lane = threadIdx.x, l = lane & (W - 1), row0 = lane & ~(W - 1);
    int64_t first;
    if (!row_slot<W>(nslot, first)) return;
    const TileDev& T = a.tiles[a.gtile[(slot0 + first) >> 6]];
    const int p = a.slot[slot0 + first + lane / W];
    int64_t eb = -1;
    int stop = -1, ci = 1, cj = 1, ck = 1;
    bool out = false;
    if (p >= 0) {
        eb = B.base[T.base + p] - B.e0;
        if (eb >= 0 && eb < B.ne) {
            stop = B.stop[T.base + p];
            ci = T.pi[p];
            cj = T.pj[p];
            ck = T.pk[p];
            out = ball_outside(T, ci, cj, ck, (int)a.rad[stop]);
        }
    }
    double* fb = B.fb + (stop >= 0 ? eb : 0) * BLK;
    double Fprev = 0.0, dFbarp = 0.0, Fn = stop >= max(l, 1) ? *entry_of(B, eb, l) : 0.0;
    for (int sb = 0; __ballot(sb <= stop) != 0ull; sb += W) {
        const int s = sb + l;
        const double F = Fn;
        if (s + W <= stop) Fn = *entry_of(B, eb, s + W);
        double dF = 0.0, Fb = 0.0;
        if (s >= 2 && s <= stop) {
            const int nin = shell_cells_in(a, T, s, ci, cj, ck, out);
            dF = nin > 0 ? F / (double)nin : 0.0;
        }
        if (sb == 0) Fprev = dFbarp = __shfl(F, row0 + 1);
        for (int j = 0; j < W; ++j) {
            const double dFbar = __shfl(dF, row0 + j);
            const int t = sb + j;
            if (t >= 2 && t <= stop) {
                const double rad3p = cube(a.rad[t - 1]), rad3 = cube(a.rad[t]);
                Fprev = (rad3p * Fprev + 0.5 * (dFbarp + dFbar) * (rad3 - rad3p)) / rad3;
                dFbarp = dFbar;
            }
            if (j == l) Fb = Fprev;
        }
        if (s <= (stop | 3) && stop >= 0) fb[s] = Fb;
    }
}

// v of lane S of each four lanes.
template <int S>
__device__ __forceinline__ double quad_of(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), S * 0x55, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), S * 0x55, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// The sum of f over shell s around cell (ci, cj, ck), in the reference's order, and the number
// of its cells inside the grid; out: some may lie outside.  No sum without f.
__device__ __forceinline__ void shell_sum(const SAArgs& a, const uint32_t* __restrict__ cell8,
                                          const TileDev& T, const float* __restrict__ f, int s,
                                          int ci, int cj, int ck, int64_t c0, bool out, double& A,
                                          int& nin) {
    const int st = a.shell_start[s - 1], nc = a.shell_count[s - 1];
    const int s1 = (int)T.s1, s2 = (int)T.s2;
    auto off = [&](uint32_t w) {
        return c0 + (byte_of(w, 0) + byte_of(w, 1) * s1 + byte_of(w, 2) * s2);
    };
    A = 0.0;
    if (out) {
        nin = 0;
        for (int c = 0; c < nc; ++c) {
            const uint32_t w = cell8[st + c];
            const int i1 = ci + byte_of(w, 0), i2 = cj + byte_of(w, 1), i3 = ck + byte_of(w, 2);
            if (i1 < 1 || i1 > T.n || i2 < 1 || i2 > T.n || i3 < 1 || i3 > T.n) continue;
            nin += 1;
            if (f) A += (double)f[off(w)];
        }
        return;
    }
    nin = nc;
    if (!f) return;
    int c = 0;
    for (; c + 8 <= nc; c += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = f[off(cell8[st + c + u])];
#pragma unroll
        for (int u = 0; u < 8; ++u) A += (double)v[u];
    }
    if (c < nc) {  // up to seven more, loaded together
        float v[7];
#pragma unroll
        for (int u = 0; u < 7; ++u) v[u] = f[off(cell8[st + min(c + u, nc - 1)])];
#pragma unroll
        for (int u = 0; u < 7; ++u)
            if (c + u < nc) A += (double)v[u];
    }
}

// Sbar and Sbar2 of the collapsed peaks: the sums of psi_1 (from the profile) and psi_2 over
// shells 1 .. mc - 1, added shell by shell, over their cells.  The psi_2 sums are needed here
// only and up to there, so they are gathered here rather than with every shell of every peak:
// four lanes per peak and component (workgroup y), a shell each (one lane per peak: 3.3 -> 1.9 ms
// for the 512^3 tile; 64 peaks' psi_2 rows per wavefront did not stay in the caches, 19 % hits).
__global__ __launch_bounds__(64) void sbar_rows_kernel(SAArgs a, BlockArgs B, int64_t slot0,
                                                       int64_t nslot) {
    constexpr int W = 4;
    const int lane = threadIdx.x, q = lane & (W - 1), l = blockIdx.y;
    int64_t first;
    if (!row_slot<W>(nslot, first)) return;
    const TileDev& T = a.tiles[a.gtile[(slot0 + first) >> 6]];
    const int p = a.slot[slot0 + first + lane / W];
    int64_t eb = -1;
    int mc = 0;
    if (p >= 0) {
        eb = B.base[T.base + p] - B.e0;
        if (eb >= 0 && eb < B.ne) mc = B.cross[T.base + p];
    }
    const bool on = mc > 0;
    if (__ballot(on) == 0ull) return;
    int ci = 1, cj = 1, ck = 1;
    bool out = false;
    const float* __restrict__ e2 = l == 0 ? T.eta2x : (l == 1 ? T.eta2y : T.eta2z);
    double cS = 0.0, cT = 0.0, cN = 1.0;
    int64_t c0 = 0;
    if (on) {
        ci = T.pi[p];
        cj = T.pj[p];
        ck = T.pk[p];
        out = ball_outside(T, ci, cj, ck, (int)a.rad[mc - 1]);
        c0 = (int64_t)(ci - 1) + (cj - 1) * T.s1 + (ck - 1) * T.s2;
        cS = entry_of(B, eb, 1)[4 * BLK * (2 + l)];
        cT = T.has_eta2 ? 0.0 + (double)e2[c0] : 0.0;
    }
    for (int sb = 2; __ballot(sb <= mc - 1) != 0ull; sb += W) {
        const int s = sb + q;
        double A = 0.0, S = 0.0;
        int nin = 0;
        if (s <= mc - 1) {
            S = entry_of(B, eb, s)[4 * BLK * (2 + l)];
            shell_sum(a, B.cell8, T, T.has_eta2 ? e2 : nullptr, s, ci, cj, ck, c0, out, A, nin);
        }
        const double N = (double)nin;
        auto take = [&](double n, double sv, double av) {
            if (n > 0.0) {
                cN += n;
                cS += sv;
                cT += av;
            }
        };
        take(quad_of<0>(N), quad_of<0>(S), quad_of<0>(A));
        take(quad_of<1>(N), quad_of<1>(S), quad_of<1>(A));
        take(quad_of<2>(N), quad_of<2>(S), quad_of<2>(A));
        take(quad_of<3>(N), quad_of<3>(S), quad_of<3>(A));
    }
    if (!on || q != 0) return;
    if (cN > 0.0) {
        cS /= cN;
        cT /= cN;
    }
    const int64_t o = (int64_t)p * 3 + l;
    T.res.Sbar[o] = cS;
    T.res.Sbar2[o] = cT;
}

// ------------------------------------------------------------------ radial logic by rows
// W lanes per peak (a row): the walk's kernel_strain, eigenvalues and table lookup at shell mp
// depend on mp only, not on the shells before it, so the row evaluates W shells at once and
// takes the first that collapses.  The walk needs the strain alone; what else a collapsed peak's
// record holds is worked out afterwards (finish_rows_kernel) from the two shells on either
// side of the collapse, and the formation redshift, which one halo in eight has, by
// half_rows_kernel: in one kernel the walk held 222 registers, two wavefronts per SIMD, and
// waited for its loads (512^3 tile, ms: 7.8; walk, finish and half 2.9 + 2.5 + 1.0; with four
// lanes reading a block's lines and handing them round, 2.5 + 2.1 + 0.9.  Loading the next block
// ahead costs a wavefront per SIMD: 2.7 + 2.3 + 0.8).  Four lanes for many peaks (median walk 6
// shells): two, eight and sixteen took 4, 29 and 95 % longer; sixteen where the peaks would not
// fill the CUs.

// The weights of shell mp (kernel_strain): its shells lo .. hi within [mlow, mupp] and the first
// weight; the row's range of them.
struct RowWin {
    const double* w;
    int lo, hi, rlo, rhi;
};
template <int W>
__device__ __forceinline__ RowWin row_win(const SAArgs& a, int mp, int mlow, int mupp, bool on) {
    RowWin r;
    const int mpc = on ? mp : 1;
    const int lo0 = a.kidx[3 * mpc], hi0 = a.kidx[3 * mpc + 1];
    r.w = a.kw + (a.kidx[3 * mpc + 2] - lo0);
    r.lo = on ? (mlow > lo0 ? mlow : lo0) : 0x7fff;
    r.hi = on ? (mupp < hi0 ? mupp : hi0) : -1;
    r.rlo = r.lo;
    r.rhi = r.hi;
#pragma unroll
    for (int d = 1; d < W; d <<= 1) {
        r.rlo = min(r.rlo, __shfl_xor(r.rlo, d, W));
        r.rhi = max(r.rhi, __shfl_xor(r.rhi, d, W));
    }
    return r;
}

// The lines of a block, one shell per lane of four.
template <bool STRAIN_ONLY>
struct Entry {
    double g0, g1, g2, f0, f1, f2, x0, x1, x2, y0, y1, y2, z0, z1, z2;
    __device__ __forceinline__ void load(const double* __restrict__ q) {
        if (!STRAIN_ONLY) {
            g0 = q[1];
            const double2 gb = *reinterpret_cast<const double2*>(q + 2);
            g1 = gb.x; g2 = gb.y;
            const double2 ha = *reinterpret_cast<const double2*>(q + 16);
            f0 = ha.x; f1 = ha.y;
            f2 = q[18];
        }
        x0 = q[33];
        y0 = q[49];
        z0 = q[65];
        const double2 x = *reinterpret_cast<const double2*>(q + 34);
        const double2 y = *reinterpret_cast<const double2*>(q + 50);
        const double2 z = *reinterpret_cast<const double2*>(q + 66);
        x1 = x.x; x2 = x.y;
        y1 = y.x; y2 = y.y;
        z1 = z.x; z2 = z.y;
    }
    template <int S>
    __device__ __forceinline__ void add(KS& r, const RowWin& w, int m1) const {
        const double X0 = quad_of<S>(x0), X1 = quad_of<S>(x1), X2 = quad_of<S>(x2);
        const double Y0 = quad_of<S>(y0), Y1 = quad_of<S>(y1), Y2 = quad_of<S>(y2);
        const double Z0 = quad_of<S>(z0), Z1 = quad_of<S>(z1), Z2 = quad_of<S>(z2);
        double G0 = 0, G1 = 0, G2 = 0, F0 = 0, F1 = 0, F2 = 0;
        if (!STRAIN_ONLY) {
            G0 = quad_of<S>(g0); G1 = quad_of<S>(g1); G2 = quad_of<S>(g2);
            F0 = quad_of<S>(f0); F1 = quad_of<S>(f1); F2 = quad_of<S>(f2);
        }
        if (m1 >= w.lo && m1 <= w.hi) {
            const double wt = w.w[m1], hw = 0.5 * wt;
            if (!STRAIN_ONLY) {
                r.g0 += wt * G0;
                r.g1 += wt * G1;
                r.g2 += wt * G2;
                r.f0 += wt * F0;
                r.f1 += wt * F1;
                r.f2 += wt * F2;
            }
            r.E11 -= hw * (X0 + X0);
            r.E12 -= hw * (X1 + Y0);
            r.E13 -= hw * (X2 + Z0);
            r.E22 -= hw * (Y1 + Y1);
            r.E23 -= hw * (Y2 + Z1);
            r.E33 -= hw * (Z2 + Z2);
        }
    }
};

// kernel_strain of a row: lane l's shell mp with window [mlow, mupp], for lanes with `on`; eb =
// first block of the row's peak.  The sums run over the shells in ascending order, as kstrain's.
// Four lanes read a block's lines, a shell each, and hand them round.
template <int W, bool STRAIN_ONLY>
__device__ __forceinline__ KS kstrain_row(const SAArgs& a, const BlockArgs& B, int64_t eb, int mp,
                                          int mlow, int mupp, bool on) {
    KS r = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const RowWin w = row_win<W>(a, mp, mlow, mupp, on);
    const int b1 = w.rlo <= w.rhi ? w.rhi >> 2 : -1;
    int b = w.rlo >> 2;
    Entry<STRAIN_ONLY> cur;
    const double* q = B.prof + (eb + b) * BLK_LINES + (threadIdx.x & 3) * 4;
    for (; b <= b1; ++b, q += BLK_LINES) {
        cur.load(q);
        cur.template add<0>(r, w, 4 * b);
        cur.template add<1>(r, w, 4 * b + 1);
        cur.template add<2>(r, w, 4 * b + 2);
        cur.template add<3>(r, w, 4 * b + 3);
    }
    const double sc = on && mp > 1 ? a.wRnor / a.rad[mp] : a.aRnor;
    r.E11 *= sc; r.E12 *= sc; r.E13 *= sc; r.E22 *= sc; r.E23 *= sc; r.E33 *= sc;
    if (!STRAIN_ONLY) {
        r.g0 *= sc; r.g1 *= sc; r.g2 *= sc; r.f0 *= sc; r.f1 *= sc; r.f2 *= sc;
    }
    return r;
}

__device__ __forceinline__ KS shfl_ks(const KS& k, int src) {
    KS r;
    r.E11 = __shfl(k.E11, src); r.E12 = __shfl(k.E12, src); r.E13 = __shfl(k.E13, src);
    r.E22 = __shfl(k.E22, src); r.E23 = __shfl(k.E23, src); r.E33 = __shfl(k.E33, src);
    r.g0 = __shfl(k.g0, src); r.g1 = __shfl(k.g1, src); r.g2 = __shfl(k.g2, src);
    r.f0 = __shfl(k.f0, src); r.f1 = __shfl(k.f1, src); r.f2 = __shfl(k.f2, src);
    return r;
}

// Running lapd sum over the cells of shells 1 .. sR: variants B and C from the centre on,
// skipping cells outside the grid; variant A without the centre, up to the first cell outside.
__device__ double block_d2f(const SAArgs& a, const TileDev& T, int ci, int cj, int ck, int sR) {
    const int64_t c0 = (int64_t)(ci - 1) + (cj - 1) * T.s1 + (ck - 1) * T.s2;
    const bool varA = a.variant == HNT_VARIANT_A;
    double lap = 0.0;
    int64_t n = 0;
    const int first = varA ? a.shell_start[1] : 0;
    const int last = sR >= 1 ? a.shell_start[sR - 1] + a.shell_count[sR - 1] : 0;
    for (int c = first; c < last; ++c) {
        const int4 o = a.cells[c];
        const int i1 = ci + o.x, i2 = cj + o.y, i3 = ck + o.z;
        if (i1 < 1 || i1 > T.n || i2 < 1 || i2 > T.n || i3 < 1 || i3 > T.n) {
            if (varA) break;
            continue;
        }
        lap += (double)T.lapd[c0 + o.x + o.y * T.s1 + o.z * T.s2];
        n += 1;
    }
    return n > 0 ? lap / (double)n : 0.0;
}

// What the walk leaves for a slot: the collapse between shells mc - 1 (zvir1p) and mc (zvir1), the
// walk's start m0 with its window's end, and the trace at mc - 1; mc = 0 without a collapse.
struct WalkState {
    double zvir1, zvir1p, Frhoh;
    int mc, m0, mupp0, pad;
};

template <int W>
__global__ __launch_bounds__(64) void walk_rows_kernel(SAArgs a, BlockArgs B, int64_t slot0,
                                                       int64_t nslot, WalkState* __restrict__ state) {
    const int lane = threadIdx.x, l = lane & (W - 1), row0 = lane & ~(W - 1);
    int64_t first;
    if (!row_slot<W>(nslot, first)) return;
    const int64_t sl = slot0 + first + lane / W;
    const TileDev& T = a.tiles[a.gtile[(slot0 + first) >> 6]];
    const int p = a.slot[sl];
    int64_t eb = 0;
    bool valid = p >= 0;
    if (valid) {
        eb = B.base[T.base + p] - B.e0;
        valid = eb >= 0 && eb < B.ne;
        if (!valid) eb = 0;
    }
    const int m = a.NS - 1;
    int ir2min = 0, scross = 0;
    double ZZon = 0.0, fcrit = 0.0;
    if (valid) {
        ir2min = T.ir2min[p];
        ZZon = T.ZZon ? T.ZZon[p] : T.ZZon_s;
        fcrit = T.fcrit ? T.fcrit[p] : T.fcrit_s;
        scross = B.cross[T.base + p];
    }
    const double* __restrict__ fb = B.fb + eb * BLK;

    // m0: the walk's first shell and its window (RadialShell.jl:484-554)
    int m0 = 1, mupp0 = 1;
    bool live = valid;
    if (valid) {
        m0 = first_r2_gt(a.shell_r2, 2, m, ir2min);
        if (m0 > m) m0 = m;
        bool tail = false;  // no crossing within the hunt radius
        if (fb[m0] >= fcrit) {
            if (scross > 0) m0 = scross;
            else tail = true;
        } else {
            bool found = false;
            for (int mp = m0 - 1 > 1 ? m0 - 1 : 1; mp >= 1; --mp) {
                if (fb[mp] >= fcrit) {
                    found = true;
                    break;
                }
                m0 = mp;
            }
            live = found;
        }
        mupp0 = tail ? m : B.win[3 * m0];
        if (m0 == 1) live = false;
    }
    const int mlow0 = B.win[3 * m0 + 2];

    // step i is shell m0 - 1 - i; the step before the first counts as zvir -1
    WalkState ws = {-1.0, -1.0, 0.0, 0, m0, mupp0, 0};
    double zcarry = -1.0;
    for (int i0 = 0;; i0 += W) {
        const int mp = m0 - 1 - (i0 + l);
        const bool on = live && mp >= 1;
        if (__ballot(on) == 0ull) break;
        int mlow = 1, mupp = 0;
        if (on) {
            mlow = min(mlow0, B.win[3 * mp + 2]);
            mupp = mupp0 <= B.win[3 * mp + 1] ? mupp0 : B.win[3 * mp];
        }
        const KS kk = kstrain_row<W, true>(a, B, eb, mp, mlow, mupp, on);
        double zv = -1.0, Fr = 0.0;
        if (on) {
            double lam[3], e_mp, p_mp;
            eig_ks(kk, lam);
            ev_from_lam(lam, &Fr, &e_mp, &p_mp);
            const double Fb = fb[mp];
            if (Fb > 0.0) {
                const double poe = e_mp < 1e-5 ? 0.0 : p_mp / e_mp;
                zv = interp3(a.ct, log10(Fb), e_mp, poe);
            }
        }
        const bool hit = on && zv >= ZZon;
        const uint64_t hits = (__ballot(hit) >> row0) & ((1ull << W) - 1ull);
        const int hl = hits ? __ffsll((unsigned long long)hits) - 1 : 0;
        const double zl = __shfl(zv, row0 + hl), fl = __shfl(Fr, row0 + hl);
        const double zb = __shfl(zv, row0 + (hl > 0 ? hl - 1 : 0));
        if (hits != 0 && live) {
            ws.zvir1p = zl;
            ws.Frhoh = fl;
            ws.zvir1 = hl == 0 ? zcarry : zb;
            ws.mc = m0 - (i0 + hl);
            live = false;
        }
        zcarry = __shfl(zv, row0 + W - 1);
    }
    if (!valid || l != 0) {
        if (l == 0) state[sl - slot0].mc = 0;
        return;
    }
    // RTHL > 0 (a collapse at the centre has radius 0)
    if (ws.mc > 0) {
        const double dZ = ws.zvir1p - ws.zvir1;
        double R3 = cube(a.rad[ws.mc - 1]);
        if (ws.zvir1 > 0.0 && dZ != 0.0)
            R3 = R3 + (cube(a.rad[ws.mc]) - R3) * (ws.zvir1p - ZZon) / dZ;
        if (R3 == 0.0) ws.mc = 0;
    }
    state[sl - slot0] = ws;
    if (T.res.nshells_used) T.res.nshells_used[p] = B.stop[T.base + p];
    if (T.res.crossing_shell) T.res.crossing_shell[p] = scross;
    if (T.res.bracket) T.res.bracket[p] = 0;
    B.cross[T.base + p] = ws.mc;  // what sbar_rows_kernel reads
    if (ws.mc == 0) {
        write_no_collapse(T, p);
        if (a.paint) a.paint[T.base + p] = -1;
    }
}

__device__ __forceinline__ double walk_rthl(const SAArgs& a, const WalkState& ws, double ZZon) {
    const double* rad = a.rad;
    const double dZvir = ws.zvir1p - ws.zvir1;
    if (ws.zvir1 > 0.0 && dZvir != 0.0) {
        const double RTHL3 = cube(rad[ws.mc - 1]) + (cube(rad[ws.mc]) - cube(rad[ws.mc - 1])) *
                                                        (ws.zvir1p - ZZon) / dZvir;
        return pow(RTHL3, 1.0 / 3.0);
    }
    return rad[ws.mc - 1];
}

// The record of the collapsed peaks (RadialShell.jl:608-800) but for Sbar, Sbar2 and the
// formation redshift: four lanes per peak take kernel_strain at mc - 1, at mc and at the filter
// scale.  Halos of RTHL >= 3 go to `half` (hcnt of them), slot by slot.
__global__ __launch_bounds__(64) void finish_rows_kernel(SAArgs a, BlockArgs B, int64_t slot0,
                                                         int64_t nslot,
                                                         const WalkState* __restrict__ state,
                                                         int32_t* __restrict__ half,
                                                         int32_t* __restrict__ hcnt) {
    constexpr int W = 4;
    const int lane = threadIdx.x, l = lane & (W - 1), row0 = lane & ~(W - 1);
    int64_t first;
    if (!row_slot<W>(nslot, first)) return;
    const int64_t sl = slot0 + first + lane / W;
    const TileDev& T = a.tiles[a.gtile[(slot0 + first) >> 6]];
    WalkState ws = state[sl - slot0];
    const bool on = ws.mc > 0;
    if (__ballot(on) == 0ull) return;
    const double* __restrict__ rad = a.rad;
    const int p = on ? a.slot[sl] : 0;
    const int64_t eb = on ? B.base[T.base + p] - B.e0 : 0;
    const double* __restrict__ fb = B.fb + eb * BLK;
    if (!on) ws.mc = 2;
    const int mc = ws.mc;
    const double ZZon = on ? (T.ZZon ? T.ZZon[p] : T.ZZon_s) : 0.0;
    const double RTHL = on ? walk_rthl(a, ws, ZZon) : 1.0;
    const double dZvir = ws.zvir1p - ws.zvir1;

    int mp = 1, mlow = 1, mupp = 0;
    if (on && l == 2) {
        rf_window(a, T.Rf[p], mp, mlow, mupp);
    } else if (on && l < 2) {
        mp = mc - 1 + l;
        mlow = min(B.win[3 * ws.m0 + 2], B.win[3 * mp + 2]);
        mupp = (mp == ws.m0 || ws.mupp0 <= B.win[3 * mp + 1]) ? ws.mupp0 : B.win[3 * mp];
    }
    const KS kk = kstrain_row<W, false>(a, B, eb, mp, mlow, mupp, on && l < 3);
    const KS last = shfl_ks(kk, row0), prev = shfl_ks(kk, row0 + 1);
    if (on && l == 2) {
        const int64_t o3 = (int64_t)p * 3;
        T.res.gradpkrf[o3] = kk.g0;
        T.res.gradpkrf[o3 + 1] = kk.g1;
        T.res.gradpkrf[o3 + 2] = kk.g2;
    }
    const bool halfz = on && l == 0 && a.variant != HNT_VARIANT_B && RTHL / 1.0 >= 3.0;
    {
        const uint64_t hm = __ballot(halfz);
        if (hm) {
            int at = 0;
            const int f = __ffsll((unsigned long long)hm) - 1;
            if (lane == f) at = atomicAdd(hcnt, (int)__popcll(hm));
            at = __shfl(at, f) + (int)__popcll(hm & ((1ull << lane) - 1ull));
            if (halfz) half[at] = (int32_t)(sl - slot0);
        }
    }
    if (!on || l != 0) return;

    const double RTHL3 = cube(RTHL);
    const double RTHL5 = RTHL3 * RTHL * RTHL;
    const double rad3p = cube(rad[mc - 1]);
    const double rad3 = cube(rad[mc]);
    const double drad3 = rad3 - rad3p;
    const double Fbm = fb[mc - 1], Fb0 = fb[mc];
    double Fbarx;
    KS fin;  // interpolated strain and gradients
    if (ws.zvir1 > 0.0 && drad3 != 0.0) {
        const double frac = (RTHL3 - rad3p) / drad3;
        Fbarx = Fbm + frac * (Fb0 - Fbm);
        fin.E11 = last.E11 + frac * (prev.E11 - last.E11);
        fin.E12 = last.E12 + frac * (prev.E12 - last.E12);
        fin.E13 = last.E13 + frac * (prev.E13 - last.E13);
        fin.E22 = last.E22 + frac * (prev.E22 - last.E22);
        fin.E23 = last.E23 + frac * (prev.E23 - last.E23);
        fin.E33 = last.E33 + frac * (prev.E33 - last.E33);
        fin.g0 = last.g0 + frac * (prev.g0 - last.g0);
        fin.g1 = last.g1 + frac * (prev.g1 - last.g1);
        fin.g2 = last.g2 + frac * (prev.g2 - last.g2);
        fin.f0 = last.f0 + frac * (prev.f0 - last.f0);
        fin.f1 = last.f1 + frac * (prev.f1 - last.f1);
        fin.f2 = last.f2 + frac * (prev.f2 - last.f2);
    } else {
        Fbarx = Fbm;
        fin = prev;
        fin.E11 = last.E11; fin.E12 = last.E12; fin.E13 = last.E13;
        fin.E22 = last.E22; fin.E23 = last.E23; fin.E33 = last.E33;
    }
    const double tr = fin.E11 + fin.E22 + fin.E33;
    if (tr != 0.0) {
        const double sc = Fbarx / tr;
        fin.E11 *= sc; fin.E12 *= sc; fin.E13 *= sc;
        fin.E22 *= sc; fin.E23 *= sc; fin.E33 *= sc;
    }
    double lamf[3], Frc, e_f, p_f;
    eig_ks(fin, lamf);
    ev_from_lam(lamf, &Frc, &e_f, &p_f);

    double Srb = 0.0, rad5p = 0.0;
    if (mc > 2)
        for (int s = 2; s <= mc - 1; ++s) {
            const double rad5 = pow5(rad[s]);
            Srb += 0.5 * (fb[s - 1] + fb[s]) * (rad5 - rad5p);
            rad5p = rad5;
        }
    if (ws.zvir1 > 0.0 && dZvir != 0.0) Srb += 0.5 * (Fbm + Fbarx) * (RTHL5 - rad5p);
    if (Fbarx * RTHL5 > 0.0) Srb /= (Fbarx * RTHL5);
    const int sR = first_gt(rad, 1, a.NS, RTHL) - 1;
    if (a.paint) a.paint[T.base + p] = T.mask ? a.shell_r2[sR - 1] : -1;
    double F11 = last.E11, F12 = last.E12, F13 = last.E13, F22 = last.E22, F23 = last.E23,
           F33 = last.E33;
    if (a.variant == HNT_VARIANT_A || ws.Frhoh != 0.0) {
        const double sc2 = Fbarx / ws.Frhoh;
        F11 *= sc2; F12 *= sc2; F13 *= sc2; F22 *= sc2; F23 *= sc2; F33 *= sc2;
    }
    const hnt_results& R = T.res;
    const int64_t o3 = (int64_t)p * 3;
    R.RTHL[p] = RTHL;
    R.Fbarx[p] = Fbarx;
    R.e_v[p] = e_f;
    R.p_v[p] = p_f;
    R.Srb[p] = Srb;
    R.d2F[p] = T.has_lapd ? block_d2f(a, T, T.pi[p], T.pj[p], T.pk[p], sR) : 0.0;
    // half_rows_kernel overwrites it for the halos of its list
    R.zvir_half[p] = a.variant == HNT_VARIANT_B ? 0.0 : -1.0;
    double* sm = R.strain + (int64_t)p * 9;
    sm[0] = F11; sm[1] = F12; sm[2] = F13;
    sm[3] = F12; sm[4] = F22; sm[5] = F23;
    sm[6] = F13; sm[7] = F23; sm[8] = F33;
    R.eigs[o3] = lamf[0]; R.eigs[o3 + 1] = lamf[1]; R.eigs[o3 + 2] = lamf[2];
    R.gradpk[o3] = fin.g0; R.gradpk[o3 + 1] = fin.g1; R.gradpk[o3 + 2] = fin.g2;
    R.gradpkf[o3] = fin.f0; R.gradpkf[o3 + 1] = fin.f1; R.gradpkf[o3 + 2] = fin.f2;
}

// The formation redshift (RadialShell.jl:801-859) of the listed halos: sixteen lanes per halo, ten
// of them a radius each.
__global__ __launch_bounds__(64) void half_rows_kernel(SAArgs a, BlockArgs B, int64_t slot0,
                                                       const WalkState* __restrict__ state,
                                                       const int32_t* __restrict__ half,
                                                       const int32_t* __restrict__ hcnt) {
    constexpr int W = 16, NR = 64 / W;
    const int lane = threadIdx.x, l = lane & (W - 1);
    const int n = *hcnt, m = a.NS - 1;
    const double* __restrict__ rad = a.rad;
    for (int i0 = (int)blockIdx.x * NR; i0 < n; i0 += (int)gridDim.x * NR) {
        const int i = i0 + lane / W;
        const bool row = i < n;
        const int64_t sl = slot0 + half[row ? i : i0];
        const TileDev& T = a.tiles[a.gtile[sl >> 6]];
        const int p = a.slot[sl];
        const int64_t eb = B.base[T.base + p] - B.e0;
        const double* __restrict__ fb = B.fb + eb * BLK;
        const WalkState ws = state[sl - slot0];
        const double RTHL = walk_rthl(a, ws, T.ZZon ? T.ZZon[p] : T.ZZon_s);
        const bool on = row && l < 10;
        int mp = 1, mlow = 1, mupp = 0;
        if (on) {
            const double rcur = RTHL * pow((double)l / 9.0 * 0.5 + 0.5, 1.0 / 3.0);
            mupp = 1;
            if (m - 1 >= 2) {
                const int f = first_gt(rad, 2, m - 1, rcur + 2.0);
                mupp = f <= m - 1 ? f : m - 1;
            }
            double rl = rcur - 2.0;
            if (rl < 0.0) rl = 0.0;
            const int fl = first_gt(rad, 1, m - 1, rl);
            mlow = fl <= m - 1 ? fl : 1;
            if (m - 1 >= 1) {
                const int f = first_gt(rad, 1, m - 1, rcur);
                mp = f <= m - 1 ? f : m - 1;
            }
        }
        const KS kr = kstrain_row<W, true>(a, B, eb, mp, mlow, mupp, on);
        double zh = -1.0;
        if (on) {
            double lam[3], Fr, ev, pv;
            eig_ks(kr, lam);
            ev_from_lam(lam, &Fr, &ev, &pv);
            const double Fb = fb[mp];
            const double poe = ev < 1e-5 ? 0.0 : pv / ev;
            double zr = -1.0;
            if (Fb > 0.0) zr = interp3(a.ct, log10(Fb), ev, poe);
            const double zs = zr - 1.0;
            if (zs > zh) zh = zs;
        }
#pragma unroll
        for (int d = 1; d < W; d <<= 1) {
            const double o = __shfl_xor(zh, d, W);
            if (o > zh) zh = o;
        }
        if (row && l == 0) T.res.zvir_half[p] = zh;
    }
}

// ------------------------------------------------------------------ crossing pass by rows
// The crossing pass: W lanes per peak, each summing one shell's delta, W shells at a time; the
// Fbar recurrence then runs over their sums in order (every lane alike).  The same sums and
// recurrence as crossing_kernel, which keeps a lane per peak: there a wavefront's 64 peaks walk
// 64 different cache lines for every cell and lose them before the next cell (57 % hits), and it
// runs as long as its deepest peak.  Four lanes: 512^3 tile 4.2 -> 2.8 ms; two and eight were
// 12 and 7 % slower than four (a row idles beyond the crossing, at shell 7 to 12 on average);
// sixteen for few peaks, where the time is one deep peak's chain of cells.
template <int W>
__global__ __launch_bounds__(64) void crossing_rows_kernel(SAArgs a,
                                                           const uint32_t* __restrict__ cell8,
                                                           int32_t* __restrict__ stop_out,
                                                           int32_t* __restrict__ cross_out) {
    const int lane = threadIdx.x, l = lane & (W - 1), row0 = lane & ~(W - 1);
    int64_t s0;
    if (!row_slot<W>(a.ngroups * 64, s0)) return;
    const TileDev& T = a.tiles[a.gtile[s0 >> 6]];
    const int p = a.slot[s0 + lane / W];
    const bool valid = p >= 0;
    const int m = a.NS - 1;
    int ci = 1, cj = 1, ck = 1, ir2min = 0;
    double fcrit = 0.0, Rf = 0.0;
    if (valid) {
        ci = T.pi[p];
        cj = T.pj[p];
        ck = T.pk[p];
        ir2min = T.ir2min[p];
        Rf = T.Rf[p];
        fcrit = T.fcrit ? T.fcrit[p] : T.fcrit_s;
    }
    const int64_t c0 = (int64_t)(ci - 1) + (cj - 1) * T.s1 + (ck - 1) * T.s2;
    double Fprev = valid ? (double)T.delta[c0] : 0.0;
    double dFbarp = Fprev;
    bool active = valid, past = false;
    int scross = 0;
    for (int sb = 2; sb <= m; sb += W) {
        if (__ballot(active) == 0ull) break;
        const int s = sb + l;
        double F = 0.0;
        int nin = 0;
        // the shells of this batch that leave the grid are summed with the check
        const bool out = ball_outside(T, ci, cj, ck, (int)a.rad[min(sb + W - 1, m)]);
        if (active && s <= m) {
            shell_sum(a, cell8, T, T.delta, s, ci, cj, ck, c0, out, F, nin);
        }
        for (int j = 0; j < W && sb + j <= m; ++j) {
            const double Fj = __shfl(F, row0 + j);
            const int nj = __shfl(nin, row0 + j);
            if (active)
                cross_step(a, sb + j, Fj, nj, ir2min, fcrit, Fprev, dFbarp, past, active, scross);
        }
    }
    if (!valid || l != 0) return;
    stop_out[T.base + p] = crossing_stop(a, Rf, scross);
    cross_out[T.base + p] = scross;
}

// What the gather of a call amounts to, from `ns` of its peaks: per workgroup the cells within
// BR_H, from there to 20 cells, beyond, those of the peaks whose balls leave the grid, the shells
// (sums over the samples), and the largest ball's cells.  With them what else the host looks at: the
// number of blocks and of bricks.
constexpr int WK_WG = 64, WK_N = 6;
struct WorkSample {
    double v[WK_WG][WK_N];
    int64_t blocks, bricks;
};

__global__ __launch_bounds__(256) void work_sample_kernel(SAArgs a, const uint64_t* __restrict__ keys,
                                                          const int32_t* __restrict__ vals,
                                                          const int32_t* __restrict__ stop,
                                                          const int64_t* __restrict__ off,
                                                          const int32_t* __restrict__ cnt,
                                                          const int32_t* __restrict__ bricks,
                                                          int64_t ntot, int64_t ns, int near, int mid,
                                                          WorkSample* __restrict__ out) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        out->blocks = off[ntot - 1] + cnt[ntot - 1];
        out->bricks = *bricks;
    }
    double v[WK_N] = {0, 0, 0, 0, 0, 0};
    auto cells_to = [&](int s) { return (double)(a.shell_start[s - 1] + a.shell_count[s - 1]); };
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < ns; i += (int64_t)WK_WG * 256) {
        const int64_t q = i * ntot / ns, id = vals[q];
        const TileDev& T = a.tiles[keys[q] >> 50];
        const int p = (int)(id - T.base), s = stop[id];
        const double all = cells_to(s), n8 = cells_to(min(s, near)), n20 = cells_to(min(s, mid));
        if (ball_outside(T, T.pi[p], T.pj[p], T.pk[p], (int)a.rad[s])) v[3] += all;
        else {
            v[0] += n8;
            v[1] += n20 - n8;
            v[2] += all - n20;
        }
        v[4] += (double)s;
        v[5] = fmax(v[5], all);
    }
    __shared__ double part[4][WK_N];
#pragma unroll
    for (int c = 0; c < WK_N; ++c) {
        for (int d = 1; d < 64; d <<= 1) {
            const double o = __shfl_xor(v[c], d);
            v[c] = c == 5 ? fmax(v[c], o) : v[c] + o;
        }
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][c] = v[c];
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c < WK_N) {
        const double x = part[0][c], y = part[1][c], z = part[2][c], w = part[3][c];
        out->v[blockIdx.x][c] = c == 5 ? fmax(fmax(x, y), fmax(z, w)) : x + y + z + w;
    }
}

// Whether the lane-per-peak kernel is the quicker one.  v: the work (work_sample_kernel's, of the
// whole call); np peaks in nbricks bricks, tiles of ncell cells.  Its lanes share the lines
// that neighbouring peaks read, so that its cost per cell falls with the peaks' density, but it
// runs as long as its deepest peak; the far gather's cells cost the same at any density.  Milliseconds
// fitted to 100 calls (40^3 to 1024^3 cells, 3000 to 21 M peaks, hunt radii 4 to 45); blocks and
// lanes measured, of 256^3 tiles with 1 M peaks none of which crosses (all gathered to the hunt
// radius): radius 12 118 / 127, 16 354 / 291, 20 757 / 534, 30 2879 / 1654; 100 k peaks, 30: 434 /
// 280; a 1024^3 tile's own 21 M peaks 210 / 327.  Where the rule errs on those 100 it loses at most
// 13 %.  In a brick of more than 0.6 peaks a cell the items of all its peaks are listed and summed
// by one workgroup, one after another (1 M peaks of a 64^3 tile: 43 / 8.0).
bool lanes_quicker(const double* v, double np, double nbricks, double ncell) {
    const double rho = np / (4096.0 * nbricks), thin = std::pow(rho, -0.25);
    const double all = v[0] + v[1] + v[2] + v[3];
    const double lanes = 0.82e-3 * v[5] +
                         1e-6 * ((7.3e-3 + 3.8e-3 * thin) * all + 0.062 * thin * v[4] + 0.035 * ncell);
    const double blocks = 2.2 + 1e-6 * (6.2e-3 * v[0] + (21e-3 + 1.7e-3 * thin) * v[1] +
                                        (15e-3 + 9e-3 * thin) * v[2] + 51e-3 * v[3] + 1.4 * np);
    return rho > 0.6 || lanes < blocks;
}

// Chunk boundaries of a schedule too large for one profile buffer: boundary c is the start
// (sorted position) of the brick holding the first peak whose profile begins at or after
// block c * cap; out[2 c] the position, out[2 c + 1] its first block.
__global__ void chunk_bounds_kernel(const uint64_t* __restrict__ keys,
                                    const int64_t* __restrict__ off, int64_t ntot, int shift,
                                    int64_t cap, int nchunk, int64_t* __restrict__ out) {
    const int c = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (c >= nchunk) return;
    int64_t lo = 0, hi = ntot;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (off[mid] < (int64_t)c * cap) lo = mid + 1;
        else hi = mid;
    }
    if (lo < ntot) {
        const uint64_t brick = keys[lo] >> shift;
        int64_t l2 = 0, h2 = lo;
        while (l2 < h2) {
            const int64_t mid = (l2 + h2) >> 1;
            if ((keys[mid] >> shift) < brick) l2 = mid + 1;
            else h2 = mid;
        }
        lo = l2;
    }
    out[2 * c] = lo;
    out[2 * c + 1] = lo < ntot ? off[lo] : -1;
}
