// Combine stage of the scan->map path on gfx950 (reference Gvom.combine_maps,
// scripts/gvom.py:222-393).
//
// Launch sequence (stream-ordered, no host synchronisation):
//   tables    eight voxels of a z-contiguous column per lane: for each voxel, union of
//             the filled slots' occupancy (slot order) and sum of their free passes, then
//             the previous combined map with its <= 10-pass carry-over rule
//             (gvom.py:1010-1063).  Writes OCC | source-mask or the pass count, and
//             the column's occupied count.
//   scan      exclusive scan of the column counts -> first cell id of each column,
//             so ids follow the z-contiguous voxel order (a legal permutation of the
//             reference's atomic order); large maps only.
//   cells     one thread per occupied voxel: its id, the sources' records merged in
//             slot order then the previous map (gvom.py:889-980), eigenvalues
//             (1424-1487), heights (561-576).
//   maps2d    16x16 column tiles with a 15-cell halo in LDS: slope and roughness
//             (718-805), guessed height delta (593-714), positive/negative obstacle
//             and visibility maps (445-555).
//   commit    ping-pong parity of the combined buffers, set by the cell pass as
//             parity_next and made the parity by the 2D maps, and the new map's cell
//             count, written by the cell pass.
#include <hip/hip_runtime.h>

#include "gvom_cell_walk.h"
#include "gvom_kernels.h"


namespace {

constexpr uint32_t MASK31 = 0x7FFFFFFFu;
constexpr int LAST_BIT = 30;   // source-mask bit of the previous combined map

__device__ __forceinline__ float py_maxf(float a, float b) { return (b > a) ? b : a; }
__device__ __forceinline__ float py_minf(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ double py_max(double a, double b) { return (b > a) ? b : a; }
__device__ __forceinline__ double py_min(double a, double b) { return (b < a) ? b : a; }

// ------------------------------------------------------------------------------------
// Table pass.  A wavefront combines cpw consecutive columns, zl lanes per column, eight
// consecutive voxels per lane (zl = ceil(z_size / 8), cpw = 64 / zl: 8 columns at z_size 64).
// A source is the lane's own index plus one uniform offset, so its eight words come from two
// 16-byte loads (4-byte aligned: the offset is any number of voxels) and one address; lanes
// whose column or heights are off the source's map read a page of zeros, and where the shift
// in z leaves a column's ends partly off the map the words are masked.  Per word and source
// the arithmetic is one funnel shift (the sign bits collect the source mask) and a max-add.
//
// Bound by the reads: 256 x 256 x 64 with 8 slots (168 MB) takes 27.1 us, 6.2 TB/s, where a large
// copy reaches 5.2 and one that stays in the Infinity Cache 8.4; 512 x 512 x 64 (671 MB) 129 us.
// Before, a lane per voxel with four-byte loads issued about 16 vector instructions per word,
// most of them to form and select its address: 29.3 and 133 us, and 40.0 us for 250 x 250 x 60
// with 4 slots and 31.9 for 151 x 151 x 100 with 3 (18.4 and 13.1 now), whose sides, no multiple
// of 8, took a slower kernel.
constexpr int ZPL = 8;           // voxels per lane
constexpr int SRC_GROUP = 4;     // sources loaded together
constexpr int ZERO_PAGE_WORDS = 64;
static_assert(ZPL == 8, "two 16-byte loads, one byte of occupancy bits per lane");
static_assert(ZPL - 1 <= TABLE_PAD && ZPL <= ZERO_PAGE_WORDS, "a lane's loads stay inside the padded tables");

// four words at a 4-byte aligned address
typedef int32_t words4 __attribute__((ext_vector_type(4), aligned(4)));

struct Words8 {
    words4 a, b;
    __device__ __forceinline__ int32_t get(int j) const { return j < 4 ? a[j] : b[j - 4]; }
};

__device__ __forceinline__ Words8 load8(const int32_t *p) {
    Words8 w;
    w.a = *reinterpret_cast<const words4 *>(p);
    w.b = *reinterpret_cast<const words4 *>(p + 4);
    return w;
}

// Wave-uniform int32 in a scalar register.
__device__ __forceinline__ int32_t uni(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__global__ __launch_bounds__(256) void k_comb_tables(Geo g, const DevState *__restrict__ st,
                                                     const int32_t *__restrict__ slot_tables,
                                                     const int32_t *__restrict__ zero_page,
                                                     int32_t *__restrict__ comb_tables,
                                                     int32_t *__restrict__ col_count,
                                                     int32_t *__restrict__ group, uint64_t *__restrict__ occ_bits,
                                                     double *__restrict__ height, double *__restrict__ inferred,
                                                     int zl, int cpw, int wave_groups) {
    // per wavefront: a byte of occupied and a byte of free bits (passes, no hit) per lane, as
    // 64-bit words of its columns
    __shared__ __align__(16) uint8_t occ_b[4][512], free_b[4][512];
    __shared__ uint32_t wave_cells[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int32_t XY = g.XY, Z = g.Z, X = (int32_t)g.X;
    const int NW = (Z + 63) >> 6;   // occupancy words per column
    const int32_t c0 = uni((int32_t)(blockIdx.x * 4 + wv) * cpw);
    reinterpret_cast<uint64_t *>(occ_b[wv])[lane] = 0ull;
    reinterpret_cast<uint64_t *>(free_b[wv])[lane] = 0ull;
    const int cl = lane / zl, zo = lane - cl * zl, z0 = zo * ZPL;
    const int32_t c = c0 + cl;
    const bool act = cl < cpw && c < X;
    const int32_t x = c / XY, y = c - x * XY;
    const uint32_t lin = (uint32_t)c * (uint32_t)Z + (uint32_t)z0;   // V < 2^31
    const int parity = uni(st->parity), cur = 1 - parity;
    const int have_last = uni(st->have_last);
    const int last_slot = uni(st->last_slot), flip = uni(st->flip);
    const double *co = st->slot_origin[last_slot];   // combined origin = newest slot's (gvom.py:229)

    uint32_t M[ZPL], P[ZPL];
#pragma unroll
    for (int j = 0; j < ZPL; ++j) M[j] = P[j] = 0;
    // the lane's words of one source, shifted by (dx, dy, dz); reads may run up to seven words
    // past a column's ends (the tables are padded by 64 words on both sides)
    auto source = [&](const int32_t *tab, int32_t dx, int32_t dy, int32_t dz, bool use) {
        const bool ok = act & use & ((uint32_t)(x + dx) < (uint32_t)XY) & ((uint32_t)(y + dy) < (uint32_t)XY) &
                        ((uint32_t)(z0 + dz + ZPL - 1) < (uint32_t)(Z + ZPL - 1));
        const uint32_t shift = ((uint32_t)dx * (uint32_t)XY + (uint32_t)dy) * (uint32_t)Z + (uint32_t)dz;
        return load8(ok ? tab - ZPL + (lin + shift + ZPL) : zero_page);
    };
    for (int s0 = 0; s0 < g.B; s0 += SRC_GROUP) {
        Words8 v[SRC_GROUP];
        int32_t dz[SRC_GROUP];
#pragma unroll
        for (int k = 0; k < SRC_GROUP; ++k) {
            // shifts precomputed by the scan stage's commit (one 16-byte scalar load)
            const int s = s0 + k < g.B ? s0 + k : 0;
            const int4 sh = *reinterpret_cast<const int4 *>(st->comb_shift[s]);
            dz[k] = sh.z;
            v[k] = source(slot_tables + (int64_t)cur_buf(flip, s) * g.V, sh.x, sh.y, sh.z,
                          (s0 + k < g.B) & (sh.w != 0));
        }
#pragma unroll
        for (int k = 0; k < SRC_GROUP; ++k) {
            if (dz[k] == 0 && (Z & (ZPL - 1)) == 0) {   // uniform: every word is on the map
#pragma unroll
                for (int j = 0; j < ZPL; ++j) {
                    const int32_t t = v[k].get(j);
                    M[j] = __builtin_amdgcn_alignbit(M[j], (uint32_t)t, 31);   // M << 1 | sign
                    P[j] += (uint32_t)(t > 0 ? t : 0);
                }
            } else {
#pragma unroll
                for (int j = 0; j < ZPL; ++j) {
                    const int32_t t = (uint32_t)(z0 + j + dz[k]) < (uint32_t)Z ? v[k].get(j) : 0;
                    M[j] = __builtin_amdgcn_alignbit(M[j], (uint32_t)t, 31);
                    P[j] += (uint32_t)(t > 0 ? t : 0);
                }
            }
        }
    }
    // previous combined map
    const int32_t ldx = have_last ? uni((int32_t)(co[0] - st->comb_origin[parity][0])) : 0;
    const int32_t ldy = have_last ? uni((int32_t)(co[1] - st->comb_origin[parity][1])) : 0;
    const int32_t ldz = have_last ? uni((int32_t)(co[2] - st->comb_origin[parity][2])) : 0;
    const Words8 last = source(comb_tables + (int64_t)parity * g.V, ldx, ldy, ldz, have_last != 0);
    const int mshift = 32 - (g.B + SRC_GROUP - 1) / SRC_GROUP * SRC_GROUP;
    Words8 out;
    uint32_t ob = 0, fb = 0;
#pragma unroll
    for (int j = ZPL - 1; j >= 0; --j) {
        // union of the sources' occupancy and sum of their passes, then the previous map
        // (gvom.py:1010-1063); bit s of m: source s
        uint32_t m = __brev(M[j]) >> mshift, p = P[j];
        const int32_t t = (uint32_t)(z0 + j + ldz) < (uint32_t)Z ? last.get(j) : 0;
        if (t < 0) {
            if (m != 0 || p <= 10u) m |= 1u << LAST_BIT;   // carry-over (gvom.py:1058)
        } else if (m == 0) {
            p += (uint32_t)t;
        }
        int32_t o = m ? (int32_t)(GVOM_OCC | m) : (int32_t)p;
        if (j < 4) out.a[j] = o;
        else out.b[j - 4] = o;
        o = z0 + j < Z ? o : 0;
        ob = __builtin_amdgcn_alignbit(ob, (uint32_t)o, 31);
        fb = __builtin_amdgcn_alignbit(fb, 0u - (uint32_t)o, 31);   // o > 0: passes
    }
    if (act) {
        int32_t *dst = comb_tables + (int64_t)cur * g.V + lin;
        if (z0 + ZPL <= Z) {
            *reinterpret_cast<words4 *>(dst) = out.a;
            *reinterpret_cast<words4 *>(dst + 4) = out.b;
        } else {
#pragma unroll
            for (int j = 0; j < ZPL; ++j)
                if (z0 + j < Z) dst[j] = out.get(j);
        }
    }
    __syncthreads();   // the zeroed bytes
    if (act) {
        occ_b[wv][cl * (8 * NW) + zo] = (uint8_t)ob;
        free_b[wv][cl * (8 * NW) + zo] = (uint8_t)fb;
    }
    __syncthreads();
    // one lane per column
    const int32_t cc = c0 + lane;
    uint32_t cnt = 0;
    if (lane < cpw && cc < X) {
        int ff = -1;
        for (int w = 0; w < NW; ++w) {
            const uint64_t o = reinterpret_cast<const uint64_t *>(occ_b[wv])[lane * NW + w];
            const uint64_t f = reinterpret_cast<const uint64_t *>(free_b[wv])[lane * NW + w];
            occ_bits[(int64_t)cc * NW + w] = o;
            cnt += __popcll(o);
            if (ff < 0 && f) ff = w * 64 + __builtin_ctzll(f);   // lowest free voxel (gvom.py:580-590)
        }
        col_count[cc] = (int32_t)cnt;
        inferred[cc] = ff >= 0 ? ((double)ff + co[2]) * g.z_res : -1000.0;
        if (cnt == 0) {
            // no occupied voxel: the robot-radius default around the latest ego, measured to
            // the cell corner (gvom.py:561-570), else unknown (-1000); occupied columns get
            // their height from the record merge
            const int32_t xx = cc / XY, yy = cc - xx * XY;
            const double *ego = st->latest_ego;
            double h = -1000.0;
            const double xp = ((co[0] + (double)xx) * g.xy_res) - ego[0];
            const double yp = ((co[1] + (double)yy) * g.xy_res) - ego[1];
            if (xp * xp + yp * yp <= g.robot_r * g.robot_r) h = ego[2] - g.g2l;
            height[cc] = h;
        }
    }
    // the occupied voxels of the wavefront's or the block's columns
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off);
    if (wave_groups) {
        if (lane == 0 && c0 < X) group[blockIdx.x * 4 + wv] = (int32_t)cnt;
        return;
    }
    if (lane == 0) wave_cells[wv] = cnt;
    __syncthreads();
    if (threadIdx.x == 0)
        group[blockIdx.x] = (int32_t)(wave_cells[0] + wave_cells[1] + wave_cells[2] + wave_cells[3]);
}

// ------------------------------------------------------------------------------------
// Column id scan: blocks of 1024 threads scan COLSCAN consecutive column counts in place
// (exclusive, int4 loads) and write their total; k_comb_ids adds the totals of the
// earlier chunks.
constexpr int COLSCAN = gvom_plan::COLSCAN;   // 1024 threads x 4 columns
static_assert(COLSCAN == 1024 * 4, "column scan: 1024 threads x 4 columns per block");

__global__ __launch_bounds__(1024) void k_col_scan(int32_t *__restrict__ cnt, int64_t X,
                                                   int32_t *__restrict__ chunk_tot) {
    __shared__ int32_t wsum[16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t i = (int64_t)blockIdx.x * COLSCAN + 4 * t;
    // four counts per thread; past the last column they read as 0 and are not written
    int4 v = make_int4(0, 0, 0, 0);
    if (i + 3 < X) {
        v = *reinterpret_cast<const int4 *>(cnt + i);
    } else if (i < X) {
        v.x = cnt[i];
        if (i + 1 < X) v.y = cnt[i + 1];
        if (i + 2 < X) v.z = cnt[i + 2];
    }
    const int32_t sum = v.x + v.y + v.z + v.w;
    int32_t incl = sum;
    for (int off = 1; off < 64; off <<= 1) {
        int32_t u = __shfl_up(incl, off);
        if (lane >= off) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int32_t pre = incl - sum;
    for (int ww = 0; ww < w; ++ww) pre += wsum[ww];
    int4 o;
    o.x = pre;
    o.y = pre + v.x;
    o.z = o.y + v.y;
    o.w = o.z + v.z;
    if (i + 3 < X) {
        *reinterpret_cast<int4 *>(cnt + i) = o;
    } else if (i < X) {
        cnt[i] = o.x;
        if (i + 1 < X) cnt[i + 1] = o.y;
        if (i + 2 < X) cnt[i + 2] = o.z;
    }
    if (t == 1023) chunk_tot[blockIdx.x] = pre + sum;
}

// ------------------------------------------------------------------------------------
// Division of several f64 numbers by one divisor, each quotient rounded as a / b rounds it.  With
// r = 1 / b correctly rounded, one correction of a r leaves a quotient within an ulp and the next
// rounds it correctly (Markstein, IBM J. Res. Dev. 34(1), 1990), as long as the remainders do
// not underflow; here b is a count of points and |a| far from the ends of the range.  Five
// full-rate instructions instead of a division's scaling, quarter-rate reciprocal and fix-up.
struct DivideBy {
    double b, r;
    __device__ __forceinline__ explicit DivideBy(double d) : b(d), r(1.0 / d) {}
    __device__ __forceinline__ double operator()(double a) const {
        double q = a * r;
        q = fma(fma(-b, q, a), r, q);
        return fma(fma(-b, q, a), r, q);
    }
};
struct DivideByF {
    float b;
    __device__ __forceinline__ explicit DivideByF(float d) : b(d) {}
    __device__ __forceinline__ float operator()(float a) const { return a / b; }
};
template <typename T> struct DivideOf { using type = DivideByF; };
template <> struct DivideOf<double> { using type = DivideBy; };

// Record merge, __combine_metrics (gvom.py:889-980) with Numba's typing: the product of
// two combined (f32) entries is f32, everything touching an f64 operand is f64.
template <typename OT>
__device__ __forceinline__ void merge_record(float cm[10], int32_t &hit, int32_t &tot, float &mh, const OT om[10],
                                             int32_t ohit, int32_t otot, float omh) {
    using MT = decltype((float)0 * (OT)0);
    const typename DivideOf<MT>::type by(cm[9] + om[9]);
    MT mx = by(cm[0] * cm[9] + om[0] * om[9]);
    MT my = by(cm[1] * cm[9] + om[1] * om[9]);
    MT mz = by(cm[2] * cm[9] + om[2] * om[9]);
    float c3 = (float)by(cm[9] * cm[3] + om[9] * om[3] + cm[9] * (cm[0] - mx) * (cm[0] - mx) +
                         om[9] * (om[0] - mx) * (om[0] - mx));
    float c4 = (float)by(cm[9] * cm[4] + om[9] * om[4] + cm[9] * (cm[0] - mx) * (cm[1] - my) +
                         om[9] * (om[0] - mx) * (om[1] - my));
    float c5 = (float)by(cm[9] * cm[5] + om[9] * om[5] + cm[9] * (cm[0] - mx) * (cm[2] - mz) +
                         om[9] * (om[0] - mx) * (om[2] - mz));
    float c6 = (float)by(cm[9] * cm[6] + om[9] * om[6] + cm[9] * (cm[1] - my) * (cm[1] - my) +
                         om[9] * (om[1] - my) * (om[1] - my));
    float c7 = (float)by(cm[9] * cm[7] + om[9] * om[7] + cm[9] * (cm[1] - my) * (cm[2] - mz) +
                         om[9] * (om[1] - my) * (om[2] - mz));
    float c8 = (float)by(cm[9] * cm[8] + om[9] * om[8] + cm[9] * (cm[2] - mz) * (cm[2] - mz) +
                         om[9] * (om[2] - mz) * (om[2] - mz));
    cm[3] = c3; cm[4] = c4; cm[5] = c5; cm[6] = c6; cm[7] = c7; cm[8] = c8;
    cm[0] = (float)mx; cm[1] = (float)my; cm[2] = (float)mz;
    cm[9] = (float)(cm[9] + om[9]);
    hit = (int32_t)((uint32_t)hit + (uint32_t)ohit);
    tot = (int32_t)((uint32_t)tot + (uint32_t)otot);
    mh = py_minf(mh, omh);
}

// __calculate_eigenvalues (gvom.py:1424-1487): f32 loads, f64 arithmetic, f32 stores,
// descending order; the middle one is 3q minus the two stored extremes.
__device__ __forceinline__ void eigen3(const float m[10], float ev[3]) {
    const double PI = 3.141592653589793;
    float xx = m[3], xy = m[4], xz = m[5], yy = m[6], yz = m[7], zz = m[8];
    float p1 = xy * xy + xz * xz + yz * yz;
    double q = (double)(xx + yy + zz) / 3.0;
    if (p1 == 0) {
        ev[0] = py_maxf(xx, py_maxf(yy, zz));
        ev[2] = py_minf(xx, py_minf(yy, zz));
        ev[1] = (float)(3.0 * q - (double)ev[0] - (double)ev[2]);
    } else {
        double p2 = ((double)xx - q) * ((double)xx - q) + ((double)yy - q) * ((double)yy - q) +
                    ((double)zz - q) * ((double)zz - q) + 2.0 * (double)p1;
        double p = sqrt(p2 / 6.0);
        double B0 = ((double)xx - q) / p, B1 = (double)xy / p, B2 = (double)xz / p;
        double B3 = ((double)yy - q) / p, B4 = (double)yz / p, B5 = ((double)zz - q) / p;
        double r = B0 * (B3 * B5 - B4 * B4) - B1 * (B1 * B5 - B4 * B2) + B2 * (B1 * B4 - B3 * B2);
        r = r / 2.0;
        double phi;
        if (r <= -1) phi = PI / 3.0;
        else if (r >= 1) phi = 0.0;
        else phi = acos(r) / 3.0;
        ev[0] = (float)(q + 2.0 * p * cos(phi));
        ev[2] = (float)(q + 2.0 * p * cos(phi + (2.0 * PI / 3.0)));
        ev[1] = (float)(3.0 * q - (double)ev[0] - (double)ev[2]);
    }
}

// State of the combined map being built, by one thread: its origin = the newest slot's
// (gvom.py:229), and the ping-pong flip (gvom.py:276-316): no other thread before the next
// kernel reads these, and the 2D maps make parity_next the parity once no kernel of the combine
// reads the old one.
__device__ __forceinline__ void begin_map(DevState *st, int cur) {
    const double *co = st->slot_origin[st->last_slot];
    st->comb_origin[cur][0] = co[0];
    st->comb_origin[cur][1] = co[1];
    st->comb_origin[cur][2] = co[2];
    st->parity_next = cur;
    st->have_last = 1;
}

// k-th (from 0) set bit of m.
__device__ __forceinline__ int select_bit(uint64_t m, int k) {
    int at = 0;
    uint32_t h = (uint32_t)m;
    int n = __popc(h);
    if (k >= n) {
        k -= n;
        at = 32;
        h = (uint32_t)(m >> 32);
    }
#pragma unroll
    for (int w = 16; w > 0; w >>= 1) {
        n = __popc(h & ((1u << w) - 1u));
        if (k >= n) {
            k -= n;
            at += w;
            h >>= w;
        }
    }
    return at;
}

// Record merge of one cell of the combined map (lin: its table index, mask: its sources) and its
// eigenvalues: sources in slot order, then the previous combined map (gvom.py:280-298).  Per
// group of MERGE_GROUP slots, all source-table loads are issued, then all record loads, then
// the merges run in order, so a thread has a group's gathers in flight together.
constexpr int MERGE_GROUP = 4;

__device__ __forceinline__ void merge_cell(const Geo &g, const DevState *__restrict__ st,
                                           const int32_t *__restrict__ slot_tables,
                                           const SlotRec *__restrict__ slot_recs, int64_t ncap,
                                           const int32_t *__restrict__ ltab, const CombRec *__restrict__ lrec, int flip,
                                           int parity, const double *__restrict__ co, int64_t lin, uint32_t mask,
                                           CombRec &out) {
    float cm[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    int32_t hit = 0, tot = 0;
    float mh = 1.0f;
    for (int s0 = 0; s0 < g.B; s0 += MERGE_GROUP) {
        uint32_t sid[MERGE_GROUP];
        bool use[MERGE_GROUP];
#pragma unroll
        for (int q = 0; q < MERGE_GROUP; ++q) {
            const int s = s0 + q;
            use[q] = s < g.B && ((mask >> s) & 1u);
            const int32_t *addr = slot_tables;   // any valid word when the source is unused
            if (use[q]) {
                const int4 sh = *reinterpret_cast<const int4 *>(st->comb_shift[s]);
                addr = slot_tables + (int64_t)cur_buf(flip, s) * g.V + lin +
                       ((int64_t)sh.x * g.XY + sh.y) * g.Z + sh.z;
            }
            sid[q] = (uint32_t)*addr & MASK31;
        }
        SlotRec rec[MERGE_GROUP];
#pragma unroll
        for (int q = 0; q < MERGE_GROUP; ++q)
            rec[q] = slot_recs[(int64_t)cur_buf(flip, use[q] ? s0 + q : 0) * ncap + (use[q] ? sid[q] : 0)];
#pragma unroll
        for (int q = 0; q < MERGE_GROUP; ++q)
            if (use[q]) merge_record<double>(cm, hit, tot, mh, rec[q].m, rec[q].hit, rec[q].total, rec[q].min_h);
    }
    if (mask & (1u << LAST_BIT)) {
        const double *lo = st->comb_origin[parity];
        const int64_t dx = (int64_t)(co[0] - lo[0]), dy = (int64_t)(co[1] - lo[1]), dz = (int64_t)(co[2] - lo[2]);
        const uint32_t lid = (uint32_t)ltab[lin + (dx * g.XY + dy) * g.Z + dz] & MASK31;
        const CombRec &q = lrec[lid];
        merge_record<float>(cm, hit, tot, mh, q.m, q.hit, q.total, q.min_h);
    }
    out.hit = hit;
    out.total = tot;
    out.min_h = mh;
#pragma unroll
    for (int j = 0; j < 10; ++j) out.m[j] = cm[j];
    eigen3(cm, out.ev);
}

// Cells of the combined map, an equal share per thread whatever columns they are in: ids in z order
// from the first column on, the table entry becomes OCC | id, and the record merge of the cell:
// sources in slot order, then the previous combined map (gvom.py:280-298).  A block makes the
// first id of every group of gcols columns from the table pass's counts (a prefix sum in LDS);
// a thread finds its id's group there, the column from the group's column counts and the height
// from the column's occupancy words, so no list of cells goes through memory.  The thread holding
// a column's lowest occupied voxel writes its height (min_h + z + oz) * z_res (gvom.py:572-576).
//
// The ids are dealt out evenly because cells crowd: a wall fills whole columns, and with the cells
// of 256 fixed columns to a block the fullest block set the time.  71k cells of a scene with walls
// on 256 x 256 x 64 took 71 us that way and take 20.0 (8 slots), 204 and 48 with 30 slots, 98 and
// 26 on 256 x 256 x 256 (85k cells); an even scene's 38k cells 16.3 and 16.9, 64 x 64 x 32 9.0 and
// 9.4 (the column's counts are one more load in the chain).
//
// Bound by latency: a cell is a chain of column counts -> occupancy word -> table word -> source
// words -> records, the last two twice for eight slots, and the merges between them.  Two
// wavefronts fit a SIMD; one block of eight a compute unit gives every SIMD two and makes the
// prefix sum once there.  512 blocks of four took 20.7 and 19.2 us on the 71k and 38k cells
// above, 1024 30.5 and 19.0, 256 blocks of four 30.5 and 18.2.
constexpr int CELL_THREADS = 512;
constexpr int CELL_SCAN = 4;      // prefix sum: up to CELL_SCAN x 4 groups per thread
constexpr int CELL_BLOCKS = 256;
constexpr int CELL_MAX_GROUPS = CELL_SCAN * 4 * CELL_THREADS;

__global__ __launch_bounds__(CELL_THREADS) void k_comb_cells(
    Geo g, DevState *__restrict__ st, const int32_t *__restrict__ slot_tables, const SlotRec *__restrict__ slot_recs,
    int64_t ncap, int32_t *__restrict__ comb_tables, CombRec *__restrict__ comb_recs, int64_t ccap,
    const int32_t *__restrict__ col_count, const int32_t *__restrict__ group, int ngroups, int gcols,
    const uint64_t *__restrict__ occ_bits, double *__restrict__ height) {
    constexpr int WAVES = CELL_THREADS / 64;
    extern __shared__ uint4 first4[];   // first id of each group
    uint32_t *first = reinterpret_cast<uint32_t *>(first4);
    __shared__ uint32_t wtot[CELL_SCAN][WAVES];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int NW = (g.Z + 63) >> 6;
    const int32_t X = (int32_t)g.X;
    const int parity = st->parity, cur = 1 - parity, flip = st->flip;
    // origin of the combined map being built = newest slot's (gvom.py:229)
    const double *co = st->slot_origin[st->last_slot];
    uint4 v[CELL_SCAN];
    const uint4 *g4 = reinterpret_cast<const uint4 *>(group);
#pragma unroll
    for (int q = 0; q < CELL_SCAN; ++q) {
        // the last load may run past ngroups: the counts are padded
        const int i = 4 * (q * CELL_THREADS + t);
        v[q] = make_uint4(0, 0, 0, 0);
        if (i < ngroups) {
            v[q] = g4[i / 4];
            if (i + 1 >= ngroups) v[q].y = 0;
            if (i + 2 >= ngroups) v[q].z = 0;
            if (i + 3 >= ngroups) v[q].w = 0;
        }
    }
    uint32_t before[CELL_SCAN];   // cells of the wavefront's groups before the thread's
#pragma unroll
    for (int q = 0; q < CELL_SCAN; ++q) {
        if (q * 4 * CELL_THREADS >= ngroups) break;
        const uint32_t n = v[q].x + v[q].y + v[q].z + v[q].w;
        uint32_t p = n;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t u = __shfl_up(p, off);
            if (lane >= off) p += u;
        }
        before[q] = p - n;
        if (lane == 63) wtot[q][w] = p;
    }
    __syncthreads();
    uint32_t n = 0;
#pragma unroll
    for (int q = 0; q < CELL_SCAN; ++q) {
        if (q * 4 * CELL_THREADS >= ngroups) break;
        uint32_t at = 0;
#pragma unroll
        for (int u = 0; u < WAVES; ++u) {
            if (u == w) at = n;
            n += wtot[q][u];
        }
        at += before[q];
        const int i = q * CELL_THREADS + t;
        if (4 * i < ngroups)
            first4[i] = make_uint4(at, at + v[q].x, at + v[q].x + v[q].y, at + v[q].x + v[q].y + v[q].z);
    }
    __syncthreads();
    if (blockIdx.x == 0 && t == 0) {
        // the commit of gvom.py:276-316
        begin_map(st, cur);
        st->comb_cells[cur] = (int32_t)n;
        st->comb_total = (int32_t)n;
    }
    CombRec *crec = comb_recs + (int64_t)cur * ccap;
    const CombRec *lrec = comb_recs + (int64_t)parity * ccap;
    int32_t *ctab = comb_tables + (int64_t)cur * g.V;
    const int32_t *ltab = comb_tables + (int64_t)parity * g.V;
    int top = 1;
    while (4 * top < ngroups) top *= 4;
    // 64 ids per wavefront, the blocks' first wavefronts first: few cells are spread over all blocks
    for (uint32_t id = (w * gridDim.x + blockIdx.x) * 64 + lane; id < n; id += gridDim.x * CELL_THREADS) {
        // the cell's group: the last one whose first id is at or before it
        int gi = 0;
        for (int step = top; step > 0; step >>= 2) {
            int k = 0;
#pragma unroll
            for (int u = 1; u < 4; ++u) k += gi + u * step < ngroups && first[min(gi + u * step, ngroups - 1)] <= id;
            gi += k * step;
        }
        uint32_t r = id - first[gi];
        int32_t c = gi * gcols;
        c += cell_column(reinterpret_cast<const uint4 *>(col_count + c), gcols, X - c, r);
        const bool lowest = r == 0;
        int zw = 0;
        uint64_t o = occ_bits[(int64_t)c * NW];
        while (r >= (uint32_t)__popcll(o)) {
            r -= __popcll(o);
            o = occ_bits[(int64_t)c * NW + ++zw];
        }
        const int64_t z = zw * 64 + select_bit(o, (int)r);
        const int64_t lin = (int64_t)c * g.Z + z;
        const uint32_t mask = (uint32_t)ctab[lin] & MASK31;
        ctab[lin] = (int32_t)(GVOM_OCC | id);
        CombRec out;
        merge_cell(g, st, slot_tables, slot_recs, ncap, ltab, lrec, flip, parity, co, lin, mask, out);
        if ((int64_t)id < ccap) crec[id] = out;   // the records hold ccap cells
        if (lowest) height[c] = (((double)out.min_h + (double)z) + co[2]) * g.z_res;
    }
}

// Cell ids of a large map: one lane per column assigns ids in z order (first id of the column =
// earlier chunks' totals + in-chunk exclusive prefix), rewrites the table entry to
// OCC | id and appends (voxel, source mask) to the compact list.  Bit 31 of the list's voxel word marks the lowest occupied voxel of a column.
__global__ __launch_bounds__(256) void k_comb_ids(Geo g, DevState *__restrict__ st,
                                                  int32_t *__restrict__ comb_tables,
                                                  const int32_t *__restrict__ col_base,
                                                  const int32_t *__restrict__ chunk_tot,
                                                  const uint64_t *__restrict__ occ_bits,
                                                  uint2 *__restrict__ occ_list) {
    // One lane per column, 64 columns per wavefront.  Only the occupied voxels are touched:
    // their z positions come from the occupancy words k_comb_tables wrote.
    const int lane = threadIdx.x & 63;
    const int32_t X = (int32_t)g.X, Z = g.Z;
    const int32_t cb = uni((int32_t)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 64);
    if (cb >= X) return;
    const int cur = 1 - st->parity;
    if (cb == 0 && lane == 0) begin_map(st, cur);
    const int NW = (Z + 63) >> 6;
    int32_t *ctab = comb_tables + (int64_t)cur * g.V;
    // earlier chunks' totals (a wavefront's 64 columns lie in one chunk: 64 divides COLSCAN)
    uint32_t chunk_pre = 0;
    {
        const int32_t q = cb / COLSCAN;
        for (int32_t k = lane; k < q; k += 64) chunk_pre += (uint32_t)chunk_tot[k];
        for (int off = 32; off > 0; off >>= 1) chunk_pre += __shfl_xor(chunk_pre, off);
    }
    const int32_t c = cb + lane;
    if (c >= X) return;
    uint32_t id = chunk_pre + (uint32_t)col_base[c];
    bool lowest = true;
    for (int w = 0; w < NW; ++w) {
        uint64_t ob = occ_bits[(int64_t)c * NW + w];
        while (ob) {
            const int z = w * 64 + __builtin_ctzll(ob);
            ob &= ob - 1;
            const int32_t lin = c * Z + z;
            const int32_t v = ctab[lin];
            ctab[lin] = (int32_t)(GVOM_OCC | id);
            occ_list[id] = make_uint2((uint32_t)lin | (lowest ? 0x80000000u : 0u), (uint32_t)v & MASK31);
            lowest = false;
            ++id;
        }
    }
}

// Record merge per occupied voxel of the compact list (grid-stride) of a large map.  The thread
// holding a column's lowest occupied voxel writes its height.
__global__ __launch_bounds__(256) void k_comb_merge(Geo g, DevState *__restrict__ st,
                                                    const int32_t *__restrict__ slot_tables,
                                                    const SlotRec *__restrict__ slot_recs, int64_t ncap,
                                                    const int32_t *__restrict__ comb_tables,
                                                    CombRec *__restrict__ comb_recs, int64_t ccap,
                                                    const uint2 *__restrict__ occ_list,
                                                    const int32_t *__restrict__ chunk_tot, int64_t nchunk,
                                                    double *__restrict__ height) {
    const int cur = st->parity_next, parity = 1 - cur, flip = st->flip;
    const double *co = st->comb_origin[cur];
    const int lane = threadIdx.x & 63;
    uint32_t C = 0;
    for (int64_t k = lane; k < nchunk; k += 64) C += (uint32_t)chunk_tot[k];
    for (int off = 32; off > 0; off >>= 1) C += __shfl_xor(C, off);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the new map's cell count (the commit of gvom.py:276-316)
        st->comb_cells[cur] = (int32_t)C;
        st->comb_total = (int32_t)C;
    }
    if ((int64_t)C > ccap) C = (uint32_t)ccap;   // the compact list and records hold ccap cells
    CombRec *crec = comb_recs + (int64_t)cur * ccap;
    const CombRec *lrec = comb_recs + (int64_t)parity * ccap;
    const int32_t *ltab = comb_tables + (int64_t)parity * g.V;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < (int64_t)C; id += stride) {
        const uint2 e = occ_list[id];
        const uint32_t lin = e.x & MASK31;
        CombRec out;
        merge_cell(g, st, slot_tables, slot_recs, ncap, ltab, lrec, flip, parity, co, lin, e.y, out);
        crec[id] = out;
        if (e.x >> 31) {
            const uint32_t c = lin / (uint32_t)g.Z, z = lin - c * (uint32_t)g.Z;
            height[c] = (((double)out.min_h + (double)z) + co[2]) * g.z_res;
        }
    }
}

// ------------------------------------------------------------------------------------
constexpr int TILE = 16;
constexpr int HALO = 15;
constexpr int LT = TILE + 2 * HALO;   // 46 <= 64: one 64-bit mask per tile row / column
constexpr int TT = TILE * TILE;       // cells per tile
constexpr int MT = 3 * TT;            // threads per block: three per cell
static_assert(MT % 64 == 0 && MT <= 1024 && LT <= 64, "whole wavefronts, one 64-bit mask per tile row");

// First set bit of m within [lo, hi) (bit positions), or -1.
__device__ __forceinline__ int first_in(uint64_t m, int lo, int hi) {
    if (hi <= lo) return -1;
    uint64_t r = (m >> lo);
    if (hi - lo < 64) r &= (1ull << (hi - lo)) - 1ull;
    return r ? lo + __builtin_ctzll(r) : -1;
}

// One block of MT = 3 TILE^2 threads per TILE x TILE tile: the first TILE^2 threads run the
// slope fit of their column, the second walk the same columns' positive-obstacle windows
// (dependent table and record loads), the third run the guessed-height ring search, so the
// three latency chains overlap; the first group then writes the maps.  (With the slope fit
// and the ring search on the same threads the kernel took 21.0 us on 256 x 256 cells, event
// timed; skipping either shortened it by 3.7 and 6.6 us.)
__global__ __launch_bounds__(MT) void k_maps2d(Geo g, DevState *__restrict__ st,
                                                const double *__restrict__ height,
                                                const double *__restrict__ inferred,
                                                const int32_t *__restrict__ comb_tables,
                                                const CombRec *__restrict__ comb_recs, int64_t ccap,
                                                double *__restrict__ slope_x, double *__restrict__ slope_y,
                                                double *__restrict__ rough, double *__restrict__ delta,
                                                int32_t *__restrict__ pos, int32_t *__restrict__ neg,
                                                int32_t *__restrict__ vis, uint8_t *__restrict__ host_maps) {
    __shared__ double H[LT][LT];
    __shared__ uint64_t rowm[LT];   // bit ly set when H[lx][ly] is observed (rows: fixed x)
    __shared__ uint64_t colm[LT];   // bit lx set when H[lx][ly] is observed (columns: fixed y)
    __shared__ int32_t winpv[TT];   // window density result per column of the tile
    __shared__ double dhw[TT];      // guessed-height difference per column of the tile
    const int XY = g.XY;
    const int cur = st->parity_next;
    // the flip set by the cell pass: nothing else in this kernel reads the parity
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) st->parity = cur;
    const int bx = blockIdx.y * TILE, by = blockIdx.x * TILE;   // tile origin (x rows, y fastest)
    for (int k = threadIdx.x; k < LT * LT; k += MT) {
        int lx = k / LT, ly = k % LT;
        int gx = bx - HALO + lx, gy = by - HALO + ly;
        H[lx][ly] = (gx >= 0 && gx < XY && gy >= 0 && gy < XY) ? height[(int64_t)gx * XY + gy] : -1000.0;
    }
    __syncthreads();
    {
        // observed masks by ballot: one row and one column per wavefront and round
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        for (int r = wv; r < LT; r += MT / 64) {
            bool ro = false, co = false;
            if (lane < LT) {
                ro = H[r][lane] > -1000;
                co = H[lane][r] > -1000;
            }
            const uint64_t mr = __ballot(ro), mc = __ballot(co);
            if (lane == 0) {
                rowm[r] = mr;
                colm[r] = mc;
            }
        }
    }
    __syncthreads();
    const int cell = threadIdx.x % TT, half = threadIdx.x / TT;
    const int tx = cell / TILE, ty = cell % TILE;
    const int x0 = bx + tx, y0 = by + ty;
    const bool act = x0 < XY && y0 < XY;
    const int64_t c0 = (int64_t)x0 * XY + y0;
#define HAT(gx, gy) H[(gx) - bx + HALO][(gy) - by + HALO]
    if (half == 1) {
        // __make_positive_obstacle_map's density (gvom.py:530-555): occupied voxels with
        // hit > 10 in [floor((h + pos)/zr - oz) + 1, floor((h + robot_h)/zr - oz)]; the slope
        // test that overrides it is applied by the first half
        int32_t pvw = 0;
        if (act) {
            const double h0 = HAT(x0, y0);
            const double oz = st->comb_origin[cur][2];
            const double flo = floor(((h0 + g.pos_thr) / g.z_res) - oz);
            const double fhi = floor(((h0 + g.robot_h) / g.z_res) - oz);
            if (flo + 1 >= 0 && flo + 1 < g.Z && fhi >= 0 && fhi < g.Z) {
                const int lo = (int)flo + 1, hi = (int)fhi;
                const int32_t *col = comb_tables + (int64_t)cur * g.V + c0 * g.Z;
                const CombRec *recs = comb_recs + (int64_t)cur * ccap;
                double dens = 0.0, nn = 0.0;
                // eight voxels per round: all table words, then all records, are in flight
                // together; the sums still run in z order
                for (int z0 = lo; z0 <= hi; z0 += 8) {
                    int32_t t[8], rh[8], rt[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) t[k] = (z0 + k <= hi) ? col[z0 + k] : 0;
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        rh[k] = -1;
                        rt[k] = 0;
                        if (t[k] < 0) {
                            const CombRec &r = recs[(uint32_t)t[k] & MASK31];
                            rh[k] = r.hit;
                            rt[k] = r.total;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        if (rh[k] > 10) {
                            nn += (double)rt[k];
                            dens += (double)rh[k];
                        }
                }
                if (nn > 0.0) dens /= nn;
                pvw = (int32_t)(dens * 100.0);
            }
        }
        winpv[cell] = pvw;
        __syncthreads();
        return;
    }
    if (half == 2) {
        // __guess_height (gvom.py:593-714), its loop condition and the y_nh gating as written.
        // Each one-sided edge scan returns the first observed cell in scan order, i.e. the
        // lowest set bit of the row / column mask restricted to the scanned range (cells off
        // the map are never observed, matching the reference's bounds `continue`).
        double dh_out = 0.0;
        const double h0 = HAT(x0, y0);
        const double inf0 = act ? inferred[c0] : -1000.0;
        if (!(h0 > -1000) && !(inf0 == -1000.0)) {
            const int lx0 = x0 - bx + HALO, ly0 = y0 - by + HALO;
            bool xpd = false, xnd = false, ypd = false, ynd = false;
            double xph = -1000, xnh = -1000, yph = -1000, ynh = -1000;
            int i = 0;
            while (i < 15 && !(xnd && xnd && ypd && ynd)) {
                i += 1;
                if (!xpd) {
                    if (x0 + i < XY) {   // row x0+i, dy in [-i, i)
                        int f = first_in(rowm[lx0 + i], ly0 - i, ly0 + i);
                        if (f >= 0) { xph = H[lx0 + i][f]; xpd = true; }
                    } else xpd = true;
                }
                if (!xnd) {
                    if (x0 - i >= 0) {   // row x0-i, dy in (-i, i]
                        int f = first_in(rowm[lx0 - i], ly0 - i + 1, ly0 + i + 1);
                        if (f >= 0) { xnh = H[lx0 - i][f]; xnd = true; }
                    } else xnd = true;
                }
                if (!ypd) {
                    if (y0 + i < XY) {   // column y0+i, dx in (-i, i]
                        int f = first_in(colm[ly0 + i], lx0 - i + 1, lx0 + i + 1);
                        if (f >= 0) { yph = H[f][ly0 + i]; ypd = true; }
                    } else ypd = true;
                }
                if (!ynd) {
                    if (y0 - i >= 0) {   // column y0-i, dx in [-i, i)
                        int f = first_in(colm[ly0 - i], lx0 - i, lx0 + i);
                        if (f >= 0) { ynh = H[f][ly0 - i]; ynd = true; }
                    } else ynd = true;
                }
            }
            double mn = 1000.0, mxh = inf0;
            if (xph > -1000) { mn = py_min(xph, mn); mxh = py_max(xph, mxh); }
            if (xnh > -1000) { mn = py_min(xnh, mn); mxh = py_max(xnh, mxh); }
            if (yph > -1000) { mn = py_min(yph, mn); mxh = py_max(yph, mxh); }
            if (xnh > -1000) { mn = py_min(ynh, mn); mxh = py_max(ynh, mxh); }
            double dh = mxh - mn;
            if (dh > 0) dh_out = dh;
        }
        dhw[cell] = dh_out;
        if (act) delta[c0] = dh_out;
        __syncthreads();
        return;
    }
    // first group: lanes outside the map (partial tiles) compute on in-tile LDS only and
    // write nothing, so every lane reaches the one barrier below

    // __calculate_slope (gvom.py:718-805)
    double sx = 0.0, sy = 0.0, rg = -1.0;
    {
        const int xlo = x0 - 1 < 0 ? 0 : x0 - 1, xhi = x0 + 2 > XY ? XY : x0 + 2;
        const int ylo = y0 - 1 < 0 ? 0 : y0 - 1, yhi = y0 + 2 > XY ? XY : y0 + 2;
        int ngood = 0;
        for (int xx = xlo; xx < xhi; ++xx)
            for (int yy = ylo; yy < yhi; ++yy)
                if (HAT(xx, yy) > -1000) ++ngood;
        if (ngood >= 3) {
            // pts in window order (x outer, y inner) over observed cells, as gvom.py:736-749
            double mx = 0.0, my = 0.0, mz = 0.0;
            int i = 0;
            for (int xx = xlo; xx < xhi; ++xx)
                for (int yy = ylo; yy < yhi; ++yy) {
                    double hh = HAT(xx, yy);
                    if (hh > -1000) {
                        mx += (double)xx * g.xy_res;
                        my += (double)yy * g.xy_res;
                        mz += hh;
                        ++i;
                    }
                }
            mx /= (double)i;
            my /= (double)i;
            mz /= (double)i;
            double cxx = 0.0, cxy = 0.0, cxz = 0.0, cyy = 0.0, cyz = 0.0;
            for (int xx = xlo; xx < xhi; ++xx)
                for (int yy = ylo; yy < yhi; ++yy) {
                    double hh = HAT(xx, yy);
                    if (hh > -1000) {
                        double px = (double)xx * g.xy_res, py = (double)yy * g.xy_res;
                        cxx += (px - mx) * (px - mx);
                        cxy += (px - mx) * (py - my);
                        cxz += (px - mx) * (hh - mz);
                        cyy += (py - my) * (py - my);
                        cyz += (py - my) * (hh - mz);
                    }
                }
            double det = cxx * cyy - cxy * cxy;
            if (det != 0.0) {
                double a0 = (cyy * cxz - cxy * cyz) / det;
                double a1 = (cxx * cyz - cxy * cxz) / det;
                double m = sqrt(a0 * a0 + a1 * a1 + 1.0);
                a0 /= m;
                a1 /= m;
                double err = 0.0;
                for (int xx = xlo; xx < xhi; ++xx)
                    for (int yy = ylo; yy < yhi; ++yy) {
                        double hh = HAT(xx, yy);
                        if (hh > -1000) {
                            double px = (double)xx * g.xy_res, py = (double)yy * g.xy_res;
                            double e = (hh - mz) - (a0 * (px - mx) + a1 * (py - my));
                            err += e * e;
                        }
                    }
                err /= (double)ngood;
                if (err > 0) err = log(err);
                rg = err;
                sx = atan2(a0, 1.0 / m);
                sy = atan2(a1, 1.0 / m);
            }
        }
    }

#undef HAT
    if (act) {
        slope_x[c0] = sx;
        slope_y[c0] = sy;
        rough[c0] = rg;
    }
    // __make_positive_obstacle_map (gvom.py:516-555): slope test, else the window density
    __syncthreads();
    const double dh_out = dhw[cell];
    const double h0 = H[tx + HALO][ty + HALO];
    const int32_t pv = (sqrt(sx * sx + sy * sy) >= g.slope_thr) ? 100 : winpv[cell];
    // __make_negative_obstacle_map (506-512); __make_visability_map (445-452)
    if (act) {
        const int32_t nv = (dh_out > g.neg_thr) ? 100 : 0, vv = (h0 > -1000) ? 1 : 0;
        pos[c0] = pv;
        neg[c0] = nv;
        vis[c0] = vv;
        if (host_maps) {
            // the same four maps, [pos | neg | vis | rough], into pinned host memory
            const int64_t X = g.X;
            int32_t *hm = reinterpret_cast<int32_t *>(host_maps);
            hm[c0] = pv;
            hm[X + c0] = nv;
            hm[2 * X + c0] = vv;
            reinterpret_cast<double *>(hm + 3 * X)[c0] = rg;
        }
    }
}

// ------------------------------------------------------------------------------------
// Export: internal table -> reference layout (x fastest) and encoding.
__global__ __launch_bounds__(256) void k_export_table(Geo g, const int32_t *__restrict__ table,
                                                      int32_t *__restrict__ out) {
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.V) return;
    int64_t x = v % g.XY, y = (v / g.XY) % g.XY, z = v / g.X;
    int32_t t = table[(x * g.XY + y) * g.Z + z];
    out[v] = t < 0 ? (int32_t)((uint32_t)t & MASK31) : (int32_t)(-1 - (int64_t)t);
}

// __make_voxel_pointcloud (gvom.py:482-503), rows in cell-id order.
__global__ __launch_bounds__(256) void k_debug_voxels(Geo g, const DevState *__restrict__ st, int par,
                                                      const int32_t *__restrict__ table,
                                                      const CombRec *__restrict__ recs,
                                                      float4 *__restrict__ out) {
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.V) return;
    int32_t t = table[v];
    if (t >= 0) return;
    const int64_t id = (int64_t)((uint32_t)t & MASK31);
    int64_t z = v % g.Z, c = v / g.Z, y = c % g.XY, x = c / g.XY;
    const double *o = st->comb_origin[par];
    const CombRec &r = recs[id];
    out[2 * id] = make_float4((float)(((double)x + o[0]) * g.xy_res), (float)(((double)y + o[1]) * g.xy_res),
                               (float)(((double)z + o[2]) * g.z_res), (float)((double)r.hit / (double)r.total));
    out[2 * id + 1] = make_float4((float)r.hit, r.ev[0] - r.ev[1], r.ev[1] - r.ev[2], r.ev[2]);
}

// __make_height_map_pointcloud (gvom.py:456-468; W = 7), with the positive-obstacle map beside it
// as the node's records have it (W = 8, gvom_ros.py:176-186), and
// __make_infered_height_map_pointcloud (471-479, fed with the guessed height delta, 439-440; W =
// 3): rows of W words, row index x + y*xy.  A block's 256 rows are put together in LDS and
// written as one run of words.
template <int W>
__global__ __launch_bounds__(256) void k_debug_height(Geo g, const DevState *__restrict__ st, int par,
                                                      const double *__restrict__ height,
                                                      const double *__restrict__ rough,
                                                      const double *__restrict__ sx,
                                                      const double *__restrict__ sy,
                                                      const double *__restrict__ delta,
                                                      const int32_t *__restrict__ pos,
                                                      uint32_t *__restrict__ out) {
    __shared__ uint32_t w[256 * W];
    const int64_t base = (int64_t)blockIdx.x * 256, row = base + threadIdx.x;
    if (row < g.X) {
        const int64_t y = row / g.XY, x = row - y * g.XY, c = x * g.XY + y;
        const double *o = st->comb_origin[par];
        uint32_t *r = w + threadIdx.x * W;
        r[0] = __float_as_uint((float)(((double)x + o[0]) * g.xy_res));
        r[1] = __float_as_uint((float)(((double)y + o[1]) * g.xy_res));
        r[2] = __float_as_uint((float)((W == 3 ? delta[c] : height[c]) - g.z_res));
        if (W > 3) {
            const double a = sx[c], b = sy[c];
            r[3] = __float_as_uint((float)rough[c]);
            r[4] = __float_as_uint((float)a);
            r[5] = __float_as_uint((float)b);
            r[6] = __float_as_uint((float)sqrt(a * a + b * b));
            if (W == 8) r[7] = (uint32_t)pos[c];
        }
    }
    __syncthreads();
    const int64_t left = (g.X - base) * W, n = left < 256 * W ? left : 256 * W;
    for (int64_t k = threadIdx.x; k < n; k += 256) out[base * W + k] = w[k];
}

inline unsigned nblocks(int64_t n, int per) { return (unsigned)((n + per - 1) / per > 0 ? (n + per - 1) / per : 1); }

}  // namespace

int64_t zero_page_words() { return ZERO_PAGE_WORDS; }

static int table_lanes(const Geo &g) { return (g.Z + ZPL - 1) / ZPL; }

// The table pass counts the occupied voxels per wavefront where the cell pass then has a count of
// four columns or a multiple and at most four counts a thread to sum, per block otherwise.  Shorter
// groups shorten a cell's walk, more of them lengthen the sum (cell pass, per block and per
// wavefront): 64 x 64 x 32 (64 and 256 groups) 10.5 and 9.4 us, 128 x 128 x 32 13.2 and 11.4, 256 x
// 256 x 8 18.8 and 14.9; but 256 x 256 x 64 (2048 and 8192) 16.9 and 18.5, 151 x 151 x 100 (1426 and
// 5701) 11.1 and 12.5.
constexpr int64_t WAVE_GROUPS = 4 * CELL_THREADS;
static bool wave_groups(const Geo &g) {
    const int cpw = 64 / table_lanes(g);
    return cpw % 4 == 0 && (g.X + cpw - 1) / cpw <= WAVE_GROUPS;
}

int64_t comb_group_columns(const Geo &g) { return (wave_groups(g) ? 1 : 4) * (64 / table_lanes(g)); }
int64_t comb_groups(const Geo &g) { return (g.X + comb_group_columns(g) - 1) / comb_group_columns(g); }
int64_t comb_group_words(const Geo &g) { return (comb_groups(g) + 3) / 4 * 4; }

hipError_t launch_comb_tables(const Geo &g, DevState *st, const int32_t *slot_tables, const int32_t *zero_page,
                              int32_t *comb_tables, int32_t *col_count, int32_t *group, int64_t group_words,
                              uint64_t *occ_bits, double *height, double *inferred, hipStream_t s) {
    if (comb_group_words(g) > group_words) return hipErrorInvalidValue;
    const int zl = table_lanes(g);
    const int cpw = 64 / zl;
    k_comb_tables<<<nblocks(g.X, 4 * cpw), 256, 0, s>>>(g, st, slot_tables, zero_page, comb_tables, col_count, group,
                                                        occ_bits, height, inferred, zl, cpw, wave_groups(g));
    return hipGetLastError();
}

int64_t col_chunks(int64_t X) { return gvom_plan::col_chunks(X); }

// The parity and the other device state stay as they are (the cell pass sets them).
hipError_t launch_scan_columns(int32_t *col_count, int64_t count_words, int64_t X, int32_t *chunk_tot,
                               int64_t chunk_words, DevState *, hipStream_t s) {
    if (X < 1 || gvom_plan::col_scan_count_words(X) > count_words || gvom_plan::col_scan_chunk_words(X) > chunk_words)
        return hipErrorInvalidValue;
    k_col_scan<<<(unsigned)col_chunks(X), 1024, 0, s>>>(col_count, X, chunk_tot);
    return hipGetLastError();
}

// Maps of up to this many columns (256 x 256: CELL_MAX_GROUPS groups at the greatest height) merge
// their cells in one kernel; larger ones run the column scan, k_comb_ids and k_comb_merge.  Measured
// (rocprof, the kernels' sum, one kernel against three): 65,536 columns with 38k cells 16.9 against
// 24.1 us, with 71k 20.0 against 32.1, with 71k of 30 slots 48 against 63; 22,801 columns 10.8
// against 18.3, 4,096 9.4 against 15.2.  Past the line the one kernel would still be ahead where
// its groups fit: 102,400 columns 21.8 against 33.8, 262,144 with 74k cells 26.2 against 38.5.
constexpr int64_t CELL_MAX_COLUMNS = 65536;

bool comb_cells_direct(const Geo &g) { return g.X <= CELL_MAX_COLUMNS; }

hipError_t launch_comb_cells(const Geo &g, DevState *st, const int32_t *slot_tables, const SlotRec *slot_recs,
                             int64_t ncap, int32_t *comb_tables, CombRec *comb_recs, int64_t ccap, int32_t *col_count,
                             int64_t count_words, const int32_t *group, int64_t group_words, int32_t *chunk_tot,
                             int64_t chunk_words, const uint64_t *occ_bits, uint2 *occ_list, double *height,
                             hipStream_t s) {
    if (comb_cells_direct(g)) {
        const int64_t ng = comb_groups(g);
        // the last column counts are read four at a time as well
        if (ng > CELL_MAX_GROUPS || comb_group_words(g) > group_words || (g.X + 3) / 4 * 4 > count_words)
            return hipErrorInvalidValue;
        static_assert(CELL_MAX_COLUMNS <= 8 * CELL_MAX_GROUPS, "groups past WAVE_GROUPS have at least 8 columns (z_size 256)");
        const unsigned nb = nblocks(g.V, CELL_THREADS);   // a small map's voxels need fewer blocks
        k_comb_cells<<<nb < CELL_BLOCKS ? nb : CELL_BLOCKS, CELL_THREADS, (size_t)((ng + 3) / 4) * 16, s>>>(
            g, st, slot_tables, slot_recs, ncap, comb_tables, comb_recs, ccap, col_count, group, (int)ng,
            (int)comb_group_columns(g), occ_bits, height);
        return hipGetLastError();
    }
    if (!occ_list) return hipErrorInvalidValue;
    const hipError_t e = launch_scan_columns(col_count, count_words, g.X, chunk_tot, chunk_words, st, s);
    if (e != hipSuccess) return e;
    k_comb_ids<<<nblocks((g.X + 63) / 64, 4), 256, 0, s>>>(g, st, comb_tables, col_count, chunk_tot, occ_bits, occ_list);
    k_comb_merge<<<2048, 256, 0, s>>>(g, st, slot_tables, slot_recs, ncap, comb_tables, comb_recs, ccap, occ_list,
                                      chunk_tot, col_chunks(g.X), height);
    return hipGetLastError();
}

hipError_t launch_maps2d(const Geo &g, DevState *st, const double *height, const double *inferred,
                         const int32_t *comb_tables, const CombRec *comb_recs, int64_t ccap, double *slope_x,
                         double *slope_y, double *rough, double *delta, int32_t *pos, int32_t *neg, int32_t *vis,
                         uint8_t *host_maps, hipStream_t s) {
    dim3 grid((unsigned)((g.XY + TILE - 1) / TILE), (unsigned)((g.XY + TILE - 1) / TILE));
    k_maps2d<<<grid, MT, 0, s>>>(g, st, height, inferred, comb_tables, comb_recs, ccap, slope_x, slope_y, rough,
                                  delta, pos, neg, vis, host_maps);
    return hipGetLastError();
}


hipError_t launch_export_table(const Geo &g, const int32_t *table, int32_t *out_ref, hipStream_t s) {
    k_export_table<<<nblocks(g.V, 256), 256, 0, s>>>(g, table, out_ref);
    return hipGetLastError();
}

hipError_t launch_debug_voxels(const Geo &g, const DevState *st, const int32_t *comb_tables,
                               const CombRec *comb_recs, int64_t ccap, int parity, float *out,
                               hipStream_t s) {
    k_debug_voxels<<<nblocks(g.V, 256), 256, 0, s>>>(g, st, parity, comb_tables + (int64_t)parity * g.V,
                                                     comb_recs + (int64_t)parity * ccap, (float4 *)out);
    return hipGetLastError();
}

hipError_t launch_debug_height(const Geo &g, const DevState *st, int parity, const double *height,
                               const double *rough, const double *sx, const double *sy, const double *delta,
                               const int32_t *pos, int width, float *out, hipStream_t s) {
    const unsigned nb = nblocks(g.X, 256);
    uint32_t *o = (uint32_t *)out;
    if (width == 3)
        k_debug_height<3><<<nb, 256, 0, s>>>(g, st, parity, height, rough, sx, sy, delta, pos, o);
    else if (width == 7)
        k_debug_height<7><<<nb, 256, 0, s>>>(g, st, parity, height, rough, sx, sy, delta, pos, o);
    else if (width == 8)
        k_debug_height<8><<<nb, 256, 0, s>>>(g, st, parity, height, rough, sx, sy, delta, pos, o);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
