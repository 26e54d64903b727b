// Kernels.* operation descriptors: validation and routing of the reference's
// Swift descriptors (Sources/Popcorn/Kernels/*.swift, cited per descriptor),
// with dispatch geometry chosen for wave64 and the device's CU count.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

#include "popcorn.hpp"
#include "uncached.hpp"

namespace popcorn {
namespace {

constexpr int kBlock = 256;

int deviceCUs() {
    static thread_local int cached_dev = -1, cached_cus = 256;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return cached_cus;
    }
    if (dev != cached_dev) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0) cached_cus = cus;
        (void)hipGetLastError();
        cached_dev = dev;
    }
    return cached_cus;
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool isFloat(DataType t) { return t == DataType::f32 || t == DataType::f16 || t == DataType::bf16; }

void requireElements(const Tensor &t, int64_t n, const char *what) {
    if (n < 0) throw Error::invalidArgument(std::string(what) + ": negative size");
    if (n > 0 && !t.data) throw Error::invalidArgument(std::string(what) + ": null data pointer");
    if (t.shape.elementCount() < n)
        throw Error::tensorShapeMismatch(std::string(what) + " holds " + std::to_string(t.shape.elementCount()) +
                                         " elements; the operation reads or writes " + std::to_string(n) + ".");
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// A single dispatch whose function, bindings, constants and geometry are all
// fixed at init (the common case of the reference's DispatchKernel structs).
class FixedDispatch : public DispatchKernel {
public:
    FixedDispatch(std::string fn, std::vector<Binding> b, std::vector<std::vector<uint8_t>> c, DispatchSize ds)
        : fn_(std::move(fn)), b_(std::move(b)), c_(std::move(c)), ds_(ds) {}
    std::string functionName() const override { return fn_; }
    std::vector<Binding> tensors() const override { return b_; }
    std::vector<std::vector<uint8_t>> constants() const override { return c_; }
    DispatchSize dispatchSize(const FunctionAttributes &) const override { return ds_; }

private:
    std::string fn_;
    std::vector<Binding> b_;
    std::vector<std::vector<uint8_t>> c_;
    DispatchSize ds_;
};

DispatchSize grid1(int64_t blocks, int threads, size_t lds = 0) {
    DispatchSize d;
    d.grid = dim3((unsigned)std::max<int64_t>(blocks, 0), 1, 1);
    d.block = dim3((unsigned)threads, 1, 1);
    d.dynamicLds = lds;
    return d;
}

const char *tag(DataType t) { return name(t); }

// ---------------------------------------------------------------------------
// FlashAttention / FlashDecoding (FlashAttention.swift, FlashDecoding.swift)
// ---------------------------------------------------------------------------

// FlashDecoding partition sizing: blocks per CU to aim for (default 2) and
// the fewest keys a partition takes (default 64); POPCORN_FD_BLOCKS_PER_CU
// and POPCORN_FD_MIN_KEYS override them for tuning.
int envInt(const char *name, int lo, int hi, int dflt) {
    const char *e = std::getenv(name);
    const int v = e ? std::atoi(e) : 0;
    return v >= lo && v <= hi ? v : dflt;
}
int fdBlocksPerCU() {
    static const int v = envInt("POPCORN_FD_BLOCKS_PER_CU", 1, 64, 2);
    return v;
}
int fdMinKeys() {
    static const int v = envInt("POPCORN_FD_MIN_KEYS", 1, 4096, 64);
    return v;
}
// Waves per block of the 16-bit split-KV kernels: 0 (chosen per shape, the
// default), or forced to 4 or 8 for tuning.
int fdWaves16() {
    static const int v = envInt("POPCORN_FD_WAVES", 4, 8, 0);
    return v == 4 || v == 8 ? v : 0;
}

struct AttnDims {
    int64_t B, Nq, Nkv, Sq, Sk, Hd, cap;
};

// The split-KV launch plan: the fast kernel's lanes per key row (0 = the
// generic kernel), chunks per lane, query heads per block, head groups per
// KV head and partitions per query row.
struct FdPlan {
    int lpk = 0, cpl = 1, gmax = 1, waves = 4;
    int64_t ngroups = 1, P = 1;
    std::string suffix() const {  // "<t>_l<LPK>_c<CPL>_g<G>[_w8]" without the dtype
        return "_l" + std::to_string(lpk) + "_c" + std::to_string(cpl) + "_g" + std::to_string(gmax) +
               (waves == 8 ? "_w8" : "");
    }
    int64_t block() const { return 64 * waves; }
};

FdPlan fdPlan(DataType t, const AttnDims &d, bool alignedOk, int64_t keys) {
    FdPlan f;
    const int64_t G = d.Nq / d.Nkv;
    const int kV = 16 / stride(t);
    if (alignedOk && d.Hd % kV == 0) {
        const int64_t chunks = d.Hd / kV;
        if (chunks == 8 || chunks == 16 || chunks == 32 || chunks == 64) f.lpk = (int)chunks;
        if (chunks == 128 && t == DataType::f32) {
            f.lpk = 64;
            f.cpl = 2;
        }
        if (t == DataType::f32 && chunks == 8) f.lpk = 0;  // f32 Hd 32: generic
    }
    if (f.lpk) {
        f.gmax = G <= 1 ? 1 : G <= 2 ? 2 : G <= 4 ? 4 : 8;
        if (d.Hd == 512 && f.gmax > 4) f.gmax = 4;  // 4 waves x G x Hd f32 of LDS stays <= 32 KB
    }
    f.ngroups = cdiv(G, f.gmax);
    // Partitions: enough blocks to cover every CU fdBlocksPerCU() times,
    // but at least fdMinKeys() keys per block (the reference fixes P = 8,
    // FlashDecoding.swift:77).
    const int64_t base = d.B * d.Nkv * f.ngroups * d.Sq;
    const int64_t want = cdiv(fdBlocksPerCU() * deviceCUs(), base);
    const int64_t maxByKeys = cdiv(std::max<int64_t>(keys, 1), fdMinKeys());
    f.P = std::clamp<int64_t>(std::min(want, maxByKeys), 1, 1024);
    // 16-bit kernels: 8 waves per block over half the partitions (the same
    // waves, each block twice the keys) when the keys set P and the 4-wave
    // grid would put more than one block on some CU. Measured at config 4
    // (68 -> 34 partitions): 6.85-7.07 us against 7.57-7.75 in the decode
    // step; where the 4-wave grid fits the CUs (B 1, 2048 keys) or P is set
    // by the CU count, 8 waves measured no faster or slower.
    if (f.lpk && t != DataType::f32) {
        const int forced = fdWaves16();
        const bool pick = forced ? forced == 8 : maxByKeys < want && base * f.P > deviceCUs();
        if (pick) {
            f.waves = 8;
            f.P = cdiv(f.P, 2);
        }
    }
    return f;
}

class FlashAttentionKernel : public Kernel {
public:
    FlashAttentionKernel(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, AttnDims d, float scale,
                         AttentionMask mask, const Tensor *position)
        : q_(q), k_(k), v_(v), out_(out), d_(d), scale_(scale), mask_(mask), hasPos_(position != nullptr) {
        if (position) pos_ = *position;
        // FlashAttention.swift:27-36
        if (d.Nkv <= 0 || d.Nq % d.Nkv != 0)
            throw Error::tensorShapeMismatch("FlashAttention query heads must be divisible by KV heads; got " +
                                             std::to_string(d.Nq) + " and " + std::to_string(d.Nkv) + ".");
        if (d.Hd > 512)
            throw Error::tensorShapeMismatch("FlashAttention head dim must be <= 512 (kernel limit); got " +
                                             std::to_string(d.Hd) + ".");
        if (d.B <= 0 || d.Nq <= 0 || d.Sq <= 0 || d.Hd <= 0 || d.Sk < 0)
            throw Error::tensorShapeMismatch("FlashAttention dimensions must be positive.");
        if (d.cap < d.Sk) throw Error::tensorShapeMismatch("FlashAttention key capacity is smaller than the key length.");
        if (mask.kind > 2) throw Error::invalidArgument("unknown attention mask kind");
        // FlashDecoding.swift:119-125 and :199-205, FlashAttention.swift:181-190,
        // extended with f16; Q, K and V share one dtype.
        if (!(q.dataType == k.dataType && k.dataType == v.dataType && isFloat(q.dataType) && isFloat(out.dataType)))
            throw Error::unsupportedDataTypeCombination(std::string("Unsupported FlashAttention data type combination: ") +
                                                        tag(q.dataType) + ", " + tag(k.dataType) + ", " + tag(out.dataType) + ".");
        requireElements(q, d.B * d.Nq * d.Sq * d.Hd, "FlashAttention q");
        requireElements(k, d.B * d.Nkv * d.cap * d.Hd, "FlashAttention k");
        requireElements(v, d.B * d.Nkv * d.cap * d.Hd, "FlashAttention v");
        requireElements(out, d.B * d.Nq * d.Sq * d.Hd, "FlashAttention out");
        if (hasPos_) {
            if (pos_.dataType != DataType::i32) throw Error::unsupportedDataTypeCombination("position tensor must be i32");
            requireElements(pos_, 1, "position");
        }
        path_ = Kernels::route(d.Sq, d.Hd, q.dataType);
        // the tiled kernel reads Q/K/V and writes O as 8- and 16-byte runs,
        // takes a fixed key length (no device-side position), addresses a
        // head's keys with 32-bit buffer offsets and tracks row maxima on
        // unscaled scores (scale > 0)
        if (path_ == Kernels::AttentionPath::tiled &&
            (hasPos_ || !aligned16(q.data) || !aligned16(k.data) || !aligned16(v.data) || !aligned16(out.data) ||
             !(out.dataType == q.dataType || out.dataType == DataType::f32) || !(scale > 0.0f) ||
             d.Sk * d.Hd * (int64_t)stride(q.dataType) >= (int64_t{1} << 31)))
            path_ = Kernels::AttentionPath::plain;
        if (path_ == Kernels::AttentionPath::tiled) {
            // Hd 128 and 256 run 16 query rows per wave (two waves per SIMD);
            // POPCORN_FA_ROWS=32 selects the 32-row kernel there (a tuning
            // override)
            const char *e = std::getenv("POPCORN_FA_ROWS");
            hdp_ = d.Hd <= 64 ? 64 : d.Hd <= 128 ? 128 : d.Hd <= 256 ? 256 : 512;
            // f32 has only the 16-row kernel (v_mfma_f32_16x16x4_f32)
            rows16_ = q.dataType == DataType::f32 || hdp_ == 512 ||
                      ((hdp_ == 128 || hdp_ == 256) && !(e && std::string(e) == "32"));
            // POPCORN_FA_PAIR_MERGE=0: paired tiles merged by the merge
            // kernel instead of the pair's second block (a tuning override)
            const char *pm = std::getenv("POPCORN_FA_PAIR_MERGE");
            pairMergeInKernel_ = !(pm && std::string(pm) == "0");
            tiledName_ = std::string(rows16_ ? "flash_attention_tiled16_" : "flash_attention_tiled_") + tag(q.dataType) +
                         "_" + tag(out.dataType) + "_d" + std::to_string(hdp_);
            mergeName_ = std::string("flash_attention_split_merge_") + tag(out_.dataType) + "_d" + std::to_string(hdp_);
            planTileSplit();
            // the Hd 512 and f32 kernels run every tile whole
            if (hdp_ != 512 && q_.dataType != DataType::f32) planRuns();
        }
        planSplit();
        planRows();
    }

    std::vector<Binding> tensors() const override {
        std::vector<Binding> b = {{q_, kRead}, {k_, kRead}, {v_, kRead}, {out_, kWrite}};
        if (hasPos_) b.push_back({pos_, kRead});
        return b;
    }

    std::string describe() const override {
        if (path_ == Kernels::AttentionPath::tiled)
            return runLength_ || (nSplit_ && !mergedPairs()) ? tiledName_ + "," + mergeName_ : tiledName_;
        if (rowTiles_) return rowsName_ + std::to_string(rowTiles_) + (rowsP_ > 1 ? "," + reduceName_ : std::string());
        return partialName_ + "," + reduceName_;
    }

    void encode(KernelCommandEncoder &enc) const override {
        if (rowTiles_) {
            encodeRows(enc);
            return;
        }
        if (path_ == Kernels::AttentionPath::tiled) {
            // TiledFlashAttentionConstants (the fields of
            // PopcornKernelTypes.h:133-144 and two more): one block per 128
            // query rows of each (batch, query head)
            TiledFlashAttentionConstants c{};
            c.B = (uint32_t)d_.B;
            c.Nq = (uint32_t)d_.Nq;
            c.Nkv = (uint32_t)d_.Nkv;
            c.Sq = (uint32_t)d_.Sq;
            c.Sk = (uint32_t)d_.Sk;
            c.Hd = (uint32_t)d_.Hd;
            c.qTilesPerHead = (uint32_t)cdiv(d_.Sq, tileRows());
            c.maskKind = mask_.kind;
            c.slidingWindow = mask_.kind == 1 ? mask_.window : -1;
            c.scale = scale_;
            c.kvStride = (uint32_t)d_.cap;
            c.splitFrom = (uint32_t)(c.qTilesPerHead - nSplit_);
            c.pairTiles = pairTiles_ ? (mergedPairs() ? 2u : 1u) : 0u;
            int64_t nSplit = nSplit_;
            if (runLength_) {
                if (encodeRuns(enc, c)) return;
                // no scratch: pairs, whose exchange the stream keeps (made
                // here unless the stream is captured), else whole tiles
                if (!mergedPairs() || (enc.capturing() && !pairExchangeHeld(enc.stream(), pairBytes()))) {
                    nSplit = 0;
                    c.splitFrom = c.qTilesPerHead;
                    c.pairTiles = 0;
                }
            }
            // one block per tile; a split tile's two halves take two, a pair
            // of tiles two in all
            const int64_t items = d_.B * d_.Nq * ((int64_t)c.qTilesPerHead + (c.pairTiles ? 0 : nSplit));
            if (!nSplit) {
                // no split tile: the partial-state arguments are never touched
                FixedDispatch fa(tiledName_,
                                 {{q_, kRead}, {k_, kRead}, {v_, kRead}, {out_, kWrite}, {q_, kRead}, {q_, kRead},
                                  {q_, kRead}},
                                 {bytesOf(c)}, grid1(items, tiledBlock()));
                enc.dispatch(fa);
                return;
            }
            if (mergedPairs()) {
                // the published part of each split tile (unnormalised O, then
                // (m, l) per row) and its ready flag, in the stream's
                // uncached pair exchange; the second block of each pair
                // merges, so no merge kernel
                const int64_t tiles = d_.B * d_.Nq * nSplit_;
                const size_t oBytes = (size_t)(tiles * 128 * hdp_) * 4;
                const PairExchange &x = pairExchange(enc.stream(), pairBytes());
                const uint64_t ticket = nextTicket();
                c.ticketLo = (uint32_t)ticket;
                c.ticketHi = (uint32_t)(ticket >> 32);
                Tensor pO(x.data, Shape({tiles * 128, hdp_}), DataType::f32);
                Tensor pML(static_cast<uint8_t *>(x.data) + oBytes, Shape({tiles * 128 * 2}), DataType::f32);
                Tensor flags(x.flags, Shape({(int64_t)PairExchange::kFlags}), DataType::u64);
                FixedDispatch fa(tiledName_,
                                 {{q_, kRead}, {k_, kRead}, {v_, kRead}, {out_, kWrite}, {pO, kReadWrite},
                                  {pML, kReadWrite}, {flags, kReadWrite}},
                                 {bytesOf(c)}, grid1(items, tiledBlock()));
                enc.dispatch(fa);
                return;
            }
            // the two parts of each split tile: unnormalised O, then (m, l) per row
            const int64_t rows = d_.B * d_.Nq * nSplit_ * 2 * 128;
            enc.withTemporaryTensor(ScratchSpec{{rows, hdp_}, DataType::f32}, [&](Tensor pO) {
                enc.withTemporaryTensor(ScratchSpec{{rows, 2}, DataType::f32}, [&](Tensor pML) {
                    FixedDispatch fa(tiledName_,
                                     {{q_, kRead}, {k_, kRead}, {v_, kRead}, {out_, kWrite}, {pO, kWrite}, {pML, kWrite},
                                      {q_, kRead}},
                                     {bytesOf(c)}, grid1(items, tiledBlock()));
                    enc.dispatch(fa);
                    FixedDispatch merge(mergeName_, {{pO, kRead}, {pML, kRead}, {out_, kWrite}}, {bytesOf(c)},
                                        grid1(d_.B * d_.Nq * nSplit_ * mergeBlocksPerTile(), kBlock));
                    enc.dispatch(merge);
                });
            });
            return;
        }
        // FlashDecoding.swift:54-73: borrow partial O, m, l; partial; combine.
        const int64_t slots = d_.B * d_.Nq * d_.Sq * P_;
        enc.withTemporaryTensor(ScratchSpec{{slots, d_.Hd}, DataType::f32}, [&](Tensor pO) {
            enc.withTemporaryTensor(ScratchSpec{{slots}, DataType::f32}, [&](Tensor pM) {
                enc.withTemporaryTensor(ScratchSpec{{slots}, DataType::f32}, [&](Tensor pL) {
                    encodeSplit(enc, pO, pM, pL);
                });
            });
        });
    }

    // Runs of key steps: O, then (m, l), of every run's 128 rows in one scratch
    // buffer. False, and nothing encoded, without it.
    bool encodeRuns(KernelCommandEncoder &enc, TiledFlashAttentionConstants c) const {
        const int64_t BH = d_.B * d_.Nq, rows = BH * runsPerHead_ * 128;
        return enc.tryTemporaryTensor(ScratchSpec{{rows, hdp_ + 2}, DataType::f32}, [&](Tensor part) {
            Tensor pO(part.data, Shape({rows, hdp_}), DataType::f32);
            Tensor pML(static_cast<float *>(part.data) + rows * hdp_, Shape({rows, 2}), DataType::f32);
            c.splitFrom = 0;
            c.pairTiles = 3;
            c.ticketLo = (uint32_t)runLength_;
            c.ticketHi = (uint32_t)runsPerHead_;
            FixedDispatch fa(tiledName_,
                             {{q_, kRead}, {k_, kRead}, {v_, kRead}, {out_, kWrite}, {pO, kWrite}, {pML, kWrite}, {q_, kRead}},
                             {bytesOf(c)}, grid1(BH * runsPerHead_, tiledBlock()));
            enc.dispatch(fa);
            FixedDispatch merge(mergeName_, {{pO, kRead}, {pML, kRead}, {out_, kWrite}}, {bytesOf(c)},
                                grid1(BH * (int64_t)c.qTilesPerHead * mergeBlocksPerTile(), kBlock));
            enc.dispatch(merge);
        });
    }

    // The split-KV path's partial (O, m, l) in f32: slots x (Hd + 2) floats.
    size_t splitScratchBytes() const { return (size_t)(d_.B * d_.Nq * d_.Sq * P_) * (size_t)(d_.Hd + 2) * 4; }

    // The split-KV path on caller-given partial buffers (no scratch borrowed):
    // O [slots, Hd], then m and l [slots] each, inside `bytes` at `scratch`.
    void encodeSplitInto(KernelCommandEncoder &enc, void *scratch, size_t bytes) const {
        const int64_t slots = d_.B * d_.Nq * d_.Sq * P_;
        if (splitScratchBytes() > bytes)
            throw Error(POPCORN_ERR_WORKSPACE_EXHAUSTED,
                        "split-KV attention needs " + std::to_string(splitScratchBytes()) +
                            " bytes of partials; the static scratch holds " + std::to_string(bytes) + ".");
        float *base = static_cast<float *>(scratch);
        Tensor pO(base, Shape({slots, d_.Hd}), DataType::f32);
        Tensor pM(base + slots * d_.Hd, Shape({slots}), DataType::f32);
        Tensor pL(base + slots * (d_.Hd + 1), Shape({slots}), DataType::f32);
        encodeSplit(enc, pO, pM, pL);
    }

    bool tiled() const { return path_ == Kernels::AttentionPath::tiled; }

    // Forces the split-KV kernels (the plain/decoding routes) whatever route
    // the shape would take.
    void useSplitPath() {
        path_ = Kernels::AttentionPath::decoding;
        rowTiles_ = 0;
    }

    void encodeSplit(KernelCommandEncoder &enc, const Tensor &pO, const Tensor &pM, const Tensor &pL) const {
        FlashDecodingPartialExtConstants pc = partialConstants(P_);
        DispatchSize ds;
        ds.grid = dim3((unsigned)P_, (unsigned)(d_.B * d_.Nkv * ngroups_), (unsigned)d_.Sq);
        ds.block = dim3((unsigned)partialBlock_, 1, 1);
        // the position binding is read only when keyLenFromPosition
        Tensor posOrDummy = hasPos_ ? pos_ : q_;
        FixedDispatch partial(partialName_,
                              {{q_, kRead}, {k_, kRead}, {v_, kRead}, {pO, kWrite}, {pM, kWrite}, {pL, kWrite},
                               {posOrDummy, kRead}},
                              {bytesOf(pc)}, ds);
        enc.dispatch(partial);
        encodeReduce(enc, pO, pM, pL, P_);
    }

    // A few query rows on the matrix cores: the partial states of rowsP_
    // partitions and their combine, or without scratch for them one partition,
    // of one row tile per block so that there are as many blocks as there can be.
    void encodeRows(KernelCommandEncoder &enc) const {
        const int64_t rows = d_.B * d_.Nq * d_.Sq, slots = rows * rowsP_;
        auto launch = [&](int64_t rowTiles, int64_t P, const Tensor &pO, const Tensor &pM, const Tensor &pL) {
            DispatchSize ds;
            ds.grid = dim3((unsigned)P, (unsigned)(d_.B * d_.Nkv * cdiv(d_.Sq * (d_.Nq / d_.Nkv), 16 * rowTiles)), 1);
            ds.block = dim3(kBlock, 1, 1);
            // with one partition the output is written and the partials are not; else the other way round
            FixedDispatch fa(rowsName_ + std::to_string(rowTiles),
                             {{q_, kRead}, {k_, kRead}, {v_, kRead}, {pO, P > 1 ? kWrite : kRead},
                              {pM, P > 1 ? kWrite : kRead}, {pL, P > 1 ? kWrite : kRead}, {out_, kWrite}},
                             {bytesOf(partialConstants(P))}, ds);
            enc.dispatch(fa);
        };
        if (rowsP_ > 1 && enc.tryTemporaryTensor(ScratchSpec{{slots, d_.Hd + 2}, DataType::f32}, [&](Tensor part) {
                float *base = static_cast<float *>(part.data);
                Tensor pO(base, Shape({slots, d_.Hd}), DataType::f32);
                Tensor pM(base + slots * d_.Hd, Shape({slots}), DataType::f32);
                Tensor pL(base + slots * (d_.Hd + 1), Shape({slots}), DataType::f32);
                launch(rowTiles_, rowsP_, pO, pM, pL);
                encodeReduce(enc, pO, pM, pL, rowsP_);
            }))
            return;
        launch(rowsP_ > 1 ? 1 : rowTiles_, 1, q_, q_, q_);
    }

    FlashDecodingPartialExtConstants partialConstants(int64_t P) const {
        FlashDecodingPartialExtConstants pc{};
        pc.B = (uint32_t)d_.B;
        pc.Nq = (uint32_t)d_.Nq;
        pc.Nkv = (uint32_t)d_.Nkv;
        pc.Sk = (uint32_t)d_.Sk;
        pc.Hd = (uint32_t)d_.Hd;
        pc.P = (uint32_t)P;
        pc.maskKind = mask_.kind;
        pc.slidingWindow = mask_.kind == 1 ? mask_.window : -1;
        pc.scale = scale_;
        pc.kvStride = (uint32_t)d_.cap;
        pc.Sq = (uint32_t)d_.Sq;
        pc.keyLenFromPosition = hasPos_ ? 1u : 0u;
        return pc;
    }

    void encodeReduce(KernelCommandEncoder &enc, const Tensor &pO, const Tensor &pM, const Tensor &pL, int64_t P) const {
        FlashDecodingReduceExtConstants rc{};
        rc.B = (uint32_t)d_.B;
        rc.Nq = (uint32_t)d_.Nq;
        rc.Hd = (uint32_t)d_.Hd;
        rc.P = (uint32_t)P;
        rc.Sq = (uint32_t)d_.Sq;
        // one block per (query row, 64-dim slice of the head)
        DispatchSize rs;
        rs.grid = dim3((unsigned)(d_.B * d_.Nq * d_.Sq), (unsigned)cdiv(d_.Hd, 64), 1);
        rs.block = dim3(kBlock, 1, 1);
        FixedDispatch reduce(reduceName_, {{pO, kRead}, {pM, kRead}, {pL, kRead}, {out_, kWrite}}, {bytesOf(rc)}, rs);
        enc.dispatch(reduce);
    }

private:
    // Key steps of 32 that query tile qt of 128 rows visits (fa_steps).
    int64_t keySteps(int64_t qt) const {
        const int64_t first = d_.Sk - d_.Sq + qt * 128, last = d_.Sk - d_.Sq + std::min(qt * 128 + 127, d_.Sq - 1);
        const int64_t hi = mask_.kind == 2 ? d_.Sk : std::min(d_.Sk, last + 1);
        const int64_t lo = mask_.kind == 1 ? std::max<int64_t>(0, first - mask_.window + 1) : 0;
        return hi > lo ? cdiv(hi - lo, 32) : 0;
    }

    // 2 to 31 query rows over 16-bit K/V in 16-byte rows: flash_attention_rows_*
    // (flash_attention_rows.hip), which reads K and V once for all the rows
    // of a KV head's query heads. Row tiles of 16 per block: as many as the
    // kernels have and the rows half fill, where blocks of 8 key steps (two
    // per wave) still fill the CUs, since then K/V traffic counts (4
    // sequences, 32 / 8 heads, Hd 128, 16 rows x 8000 keys: 4 tiles 52 us, 1
    // tile 64); else one (31 rows x 2000 keys, 8 heads on one, Hd 256: 1 tile
    // 15.3 us, 2 tiles 18.4). Partitions: one block per CU, a step per wave at
    // least (8 rows x 4104 keys, 4 KV heads: 33 partitions 12.2 us, 17 14.1,
    // 65 13.7); up to 12 steps one partition, which needs no combine (4 heads on
    // 2, Hd 64, 8 rows x 300 keys: 5.5 us, 500 keys in partitions 7.9). On the
    // one-row kernels the three calls take 507, 62.4 and 22.7 us.
    void planRows() {
        const int64_t lim = int64_t{1} << 31, G = d_.Nq / d_.Nkv, R = d_.Sq * G, cus = deviceCUs();
        const DataType t = q_.dataType;
        if (d_.Sq < 2 || d_.Sq >= 32 || hasPos_ || !(t == DataType::f16 || t == DataType::bf16) || d_.Hd % 8 != 0 ||
            !(out_.dataType == t || out_.dataType == DataType::f32) || !aligned16(q_.data) || !aligned16(k_.data) ||
            !aligned16(v_.data) || !(scale_ > 0.0f) || d_.Sk <= 0 || d_.Sk * d_.Hd * 2 >= lim ||
            d_.B * d_.Nkv * cdiv(R, 16) > 65535)
            return;
        const int64_t hdp = d_.Hd <= 64 ? 64 : d_.Hd <= 128 ? 128 : d_.Hd <= 256 ? 256 : 512;
        const int64_t keys = mask_.kind == 1 ? std::min<int64_t>(d_.Sk, std::max<int64_t>(mask_.window, 0) + d_.Sq) : d_.Sk;
        const int64_t steps = cdiv(keys, 32);
        auto blocks = [&](int64_t rt) { return d_.B * d_.Nkv * cdiv(R, 16 * rt); };
        rowTiles_ = hdp <= 128 ? 4 : hdp == 256 ? 2 : 1;
        while (rowTiles_ > 1 && (R <= 8 * rowTiles_ || blocks(rowTiles_) * cdiv(steps, 8) < cus)) rowTiles_ /= 2;
        rowsP_ = steps <= 12 ? 1 : std::clamp<int64_t>(cus / blocks(rowTiles_), 1, cdiv(steps, 4));
        if (fd_.lpk && !rowsFaster(hdp, keys, blocks(rowTiles_))) rowTiles_ = 0;
        rowsName_ = std::string("flash_attention_rows_") + tag(t) + "_" + tag(out_.dataType) + "_d" + std::to_string(hdp) +
                    "_r";
    }

    // Whether the few-row kernels, in `blocks` blocks per partition, are faster
    // than the one-row kernels: by estimates (us) fitted to both on 1600 shapes
    // (13 head layouts, 2-31 rows, 31-9000 keys, 1 and 4 sequences). The latter
    // read K and V once per row, mostly from the caches (V, MB), and grow with
    // it; the former have the longer chain of latencies, in steps per wave, and
    // at Hd 512 twice that (their registers spill 62 of 512, and a block is the
    // only one on its CU). The margins leave 4 of the shapes over 2% slower, the
    // worst 5%; the few-row kernels for all of them had 540, the worst 3.2 times
    // (8 heads on 4, us one-row and few-row: Hd 256, 2 rows x 700 keys 8.4 and
    // 11.0, 8 x 500 8.6 and 11.4, 8 x 1500 12.8 and 11.5, 31 x 200 10.5 and 9.4;
    // Hd 512, 2 x 300 10.4 and 29.4, 31 x 9000 271 and 70). Head dims that the
    // one-row kernels have only their any-dim form for are always faster here
    // (Hd 200, 6 x 500: 23 and 10; Hd 320, 6 x 500: 27 and 17).
    bool rowsFaster(int64_t hdp, int64_t keys, int64_t blocks) const {
        struct {
            double one, step1, wave1;                 // one partition: base, per step, per step of a wave
            double parts, wave, mbKeys, mbParts, margin;  // several, with a combine
        } const fits[] = {{3.3, 0.05, 0.58, 7.1, 0.67, 0.02, 1.0, 0.95},
                          {3.8, 0.16, 0.62, 7.5, 0.93, 0.05, 0.9, 0.95},
                          {4.9, 0.36, 0.95, 9.2, 1.70, 0.06, 0.5, 0.85},
                          {9.3, 1.00, 3.70, 19.4, 0.50, 0.185, 0.7, 0.75}};
        const auto &f = fits[hdp == 64 ? 0 : hdp == 128 ? 1 : hdp == 256 ? 2 : 3];
        const int64_t steps = cdiv(keys, 32), waveSteps = cdiv(cdiv(steps, rowsP_), 4), rows = d_.B * d_.Nq * d_.Sq;
        const double rowMB = (double)d_.Hd * 4e-6, g = fd_.gmax;
        const double V = (double)(d_.B * d_.Nkv * ngroups_ * d_.Sq * keys) * rowMB;
        const double perRow = 6.3 + 0.2 * g * (double)(d_.Hd / 64) + (0.015 + 0.05 * g) * V + (double)(rows * P_) * rowMB;
        if (rowsP_ == 1 && steps <= 12)
            return f.one + f.step1 * (double)steps + f.wave1 * (double)waveSteps < (hdp < 512 ? 0.95 : f.margin) * perRow;
        return f.parts + f.wave * (double)(waveSteps * rowTiles_) + f.mbKeys * (double)(blocks * keys) * rowMB +
                   f.mbParts * (double)(rows * rowsP_) * rowMB < f.margin * perRow;
    }

    // Runs (pairTiles 3): calls whose tiles leave CUs idle cut every tile's
    // key steps into runs of at most L steps, one block each, merged by the
    // merge kernel. L is the one of least estimated time,
    //   rounds x L x t + 9 us + 8 us + 0.2 us per MB of partials,
    // and runs are taken where that is under 0.9 of the whole or paired
    // tiles' time, longest block x t + 9 us (for pairs, which exchange their
    // halves, + 10 us at Hd 256 and + 4 at 64 and 128: with 10 there too, short
    // prompts took runs and got slower, 768 rows, 24 heads, Hd 64, f16 19.3 ->
    // 24.0 us), with t the time of a step (us, one block per CU; MI355X, fitted
    // to L swept over 9 shapes per dtype; over 300 more, of 768 to 16000 keys,
    // none that takes runs is over 1% slower for it). bf16, Hd 256, us before ->
    // after: 500 rows x 8692 keys, 8 heads 377 -> 68; 48 x 16000 684 -> 42; 1000
    // x 1000 43 -> 33; Hd 128, 300 x 3000, 32 heads 96 -> 46. Calls of under 768
    // keys keep the one launch that the tests of the paired and the split tiles
    // hold there, not because it is the faster: runs would take 0.33 to 1 of its
    // time (134 shapes of 32 to 767 rows and 400 to 767 keys, 0.63 on average;
    // 8 heads on 4, Hd 256, bf16, 32 x 640: 32.4 -> 12.7 us).
    void planRuns() {
        const int64_t nQT = cdiv(d_.Sq, 128), BH = d_.B * d_.Nq, cus = deviceCUs();
        if (d_.Sk < 768 || BH * nQT >= cus) return;
        const bool bf = q_.dataType == DataType::bf16;
        const double t = hdp_ == 256 ? (bf ? 1.37 : 1.04) : hdp_ == 128 ? (bf ? 0.90 : 0.71) : (bf ? 0.79 : 0.64);
        std::vector<int64_t> n;
        for (int64_t qt = 0; qt < nQT; ++qt) n.push_back(keySteps(qt));
        const int64_t most = *std::max_element(n.begin(), n.end());
        double best = (double)most * t + 9.0;
        if (pairTiles_) {
            double longest = 0.0;
            for (int64_t i = 0; i < nQT / 2; ++i) longest = std::max(longest, 0.5 * (double)(n[i] + n[nQT - 1 - i]) + 1.0);
            best = longest * t + (hdp_ == 256 ? 19.0 : 13.0);
        }
        best *= 0.9;
        for (int64_t L = 1; L < most; ++L) {
            int64_t items = 0, split = 0;
            for (int64_t s : n) {
                const int64_t runs = std::max<int64_t>(cdiv(s, L), 1);
                items += runs;
                split += runs > 1 ? runs : 0;
            }
            const double rounds = (double)cdiv(BH * items, cus);
            if (rounds > 2.0) continue;
            const double us = rounds * (double)L * t + 17.0 + 0.2 * 128.0 * 4e-6 * (double)(BH * split * hdp_);
            if (us < best) {
                best = us;
                runLength_ = L;
                runsPerHead_ = items;
            }
        }
    }

    // Causal prefill with few tiles per CU: the last query tiles see up to
    // twice the mean number of keys and, one tile per CU, set the kernel's
    // time. Tiles with more than half the largest tile's key steps run as
    // two blocks over the halves of their keys, merged by a second kernel.
    // Causal prefill with at most two tiles per CU splits tiles in two
    // (flash_attention_tiled.hip, fa_work). With at most one tile per CU a
    // head's query tiles are paired light with heavy (tile i with nQT - 1 - i)
    // and each pair runs as two blocks of equal work, when every pair splits
    // its heavy tile (x >= 1 steps in the first block); otherwise the tiles
    // with more than half the heaviest tile's steps run as two halves.
    void planTileSplit() {
        nSplit_ = 0;
        pairTiles_ = false;
        const int64_t nQT = cdiv(d_.Sq, 128);
        const int64_t tiles = d_.B * d_.Nq * nQT;
        // the Hd 512 and f32 kernels run every tile whole
        if (hdp_ == 512 || q_.dataType == DataType::f32 || mask_.kind != 0 || nQT < 4 || tiles > 2 * (int64_t)deviceCUs()) return;
        auto steps = [&](int64_t qt) { return keySteps(qt); };
        bool pairs = tiles <= (int64_t)deviceCUs();
        for (int64_t i = 0; pairs && i < nQT / 2; ++i) {
            const int64_t sa = steps(i), sb = steps(nQT - 1 - i);
            const int64_t x = (sa + sb + 1) / 2 - sa;
            pairs = x >= 1 && x < sb;
        }
        // one ready flag per split tile in the stream's pair exchange
        pairs = pairs && d_.B * d_.Nq * (nQT / 2) < (int64_t)PairExchange::kFlags;
        if (pairs) {
            pairTiles_ = true;
            nSplit_ = nQT / 2;
            return;
        }
        const int64_t most = steps(nQT - 1);
        int64_t from = nQT;
        while (from > 0 && steps(from - 1) * 2 > most) --from;
        if (most < 4 || from == nQT) return;
        nSplit_ = nQT - from;
    }

    void planSplit() {
        const DataType t = q_.dataType;
        const bool alignedOk = aligned16(q_.data) && aligned16(k_.data) && aligned16(v_.data);
        const FdPlan f = fdPlan(t, d_, alignedOk, hasPos_ ? d_.cap : d_.Sk);
        partialName_ = std::string("flash_decoding_partial_") + tag(t) + (f.lpk ? f.suffix() : std::string("_ext"));
        partialBlock_ = f.lpk ? f.block() : kBlock;
        reduceName_ = std::string("flash_decoding_reduce_") + tag(out_.dataType) + "_ext";
        ngroups_ = f.ngroups;
        P_ = f.P;
        fd_ = f;
    }

    Tensor q_, k_, v_, out_, pos_;
    AttnDims d_;
    float scale_;
    AttentionMask mask_;
    bool hasPos_;
    Kernels::AttentionPath path_ = Kernels::AttentionPath::plain;
    std::string partialName_, reduceName_, tiledName_, mergeName_;
    int64_t partialBlock_ = kBlock;
    int64_t nSplit_ = 0;
    bool pairTiles_ = false;
    int64_t runLength_ = 0, runsPerHead_ = 0;  // runs of key steps (0: none)
    int64_t rowTiles_ = 0, rowsP_ = 1;         // a few rows on the matrix cores (0: not)
    FdPlan fd_;
    std::string rowsName_;                     // up to its number of row tiles
    bool rows16_ = false;  // the 16-rows-per-wave kernel: 8 waves per 128-row tile (4 per 64 at Hd 512 and in f32)
    int64_t hdp_ = 0;      // the tiled kernel's head dim: Hd padded to 64, 128, 256 or 512
    bool tiles64() const { return hdp_ == 512 || q_.dataType == DataType::f32; }
    int64_t tiledBlock() const { return tiles64() ? 256 : rows16_ ? 512 : kBlock; }
    int64_t tileRows() const { return tiles64() ? 64 : 128; }
    // the merge kernel: HD / 4 lanes per row, so 1024 / HD of a tile's 128 rows per block
    int64_t mergeBlocksPerTile() const { return 128 * hdp_ / 1024; }
    // Paired tiles are merged inside the tiled kernels (pairTiles 2).
    bool pairMergeInKernel_ = true;
    bool mergedPairs() const { return pairTiles_ && pairMergeInKernel_; }
    // Merged pairs' published parts: O, then (m, l), of each split tile's 128 rows.
    size_t pairBytes() const { return (size_t)(d_.B * d_.Nq * nSplit_ * 128 * (hdp_ + 2)) * 4; }
    // A 64-bit value, never 0 or ~0 and distinct per launch, for the ready flags
    // of merged pairs: a counter, started from the clock so that processes
    // differ, through the splitmix64 finaliser.
    static uint64_t nextTicket() {
        static std::atomic<uint64_t> counter{(uint64_t)std::chrono::steady_clock::now().time_since_epoch().count()};
        for (;;) {
            uint64_t z = (counter.fetch_add(1, std::memory_order_relaxed) + 1) * 0x9E3779B97F4A7C15ull;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            z ^= z >> 31;
            if (z != 0 && z != ~0ull) return z;
        }
    }
    int64_t ngroups_ = 1, P_ = 1;
};

// The attention block of one decode token (DecodeAttentionConstants): the
// fresh-key split-KV partial kernel, then the same LSE combine.
class DecodeAttentionKernel : public Kernel {
public:
    explicit DecodeAttentionKernel(const Kernels::DecodeAttentionArgs &a) {
        if (!a.qkv || !a.kCache || !a.vCache || !a.out || !a.position)
            throw Error::invalidArgument("DecodeAttention needs qkv, both caches, out and position");
        qkv_ = *a.qkv;
        k_ = *a.kCache;
        v_ = *a.vCache;
        out_ = *a.out;
        pos_ = *a.position;
        if (k_.shape.rank() != 4) throw Error::tensorInvalidRank(4, k_.shape.rank());
        if (v_.shape != k_.shape) throw Error::tensorShapeMismatch("DecodeAttention K and V caches must have one shape.");
        d_.B = k_.shape[0];
        d_.Nkv = k_.shape[1];
        d_.cap = k_.shape[2];
        d_.Hd = k_.shape[3];
        d_.Nq = a.queryHeads;
        d_.Sq = 1;
        d_.Sk = d_.cap;
        if (d_.Nkv != a.kvHeads) throw Error::tensorShapeMismatch("DecodeAttention kv_heads must match the caches' dim 1.");
        if (d_.Nkv <= 0 || d_.Nq <= 0 || d_.Nq % d_.Nkv != 0)
            throw Error::tensorShapeMismatch("DecodeAttention query heads must be a positive multiple of the KV heads.");
        if (d_.B <= 0 || d_.cap <= 0 || d_.Hd <= 0 || d_.Hd % 2 != 0)
            throw Error::tensorShapeMismatch("DecodeAttention needs B, capacity > 0 and an even head dim.");
        if (a.mask.kind > 2) throw Error::invalidArgument("unknown attention mask kind");
        const DataType t = k_.dataType;
        if (!isFloat(t) || qkv_.dataType != t || v_.dataType != t || !(out_.dataType == t || out_.dataType == DataType::f32))
            throw Error::unsupportedDataTypeCombination("DecodeAttention: qkv and the caches of one float dtype, out of it or f32.");
        if (pos_.dataType != DataType::i32) throw Error::unsupportedDataTypeCombination("position tensor must be i32");
        requireElements(pos_, 1, "position");
        const int64_t rowStride = (d_.Nq + 2 * d_.Nkv) * d_.Hd;
        requireElements(qkv_, d_.B * rowStride, "DecodeAttention qkv");
        requireElements(k_, d_.B * d_.Nkv * d_.cap * d_.Hd, "DecodeAttention k_cache");
        requireElements(out_, d_.B * d_.Nq * d_.Hd, "DecodeAttention out");
        auto f32vec = [&](const Tensor *w, int64_t n, const char *what) {
            if (!w) return;
            if (w->dataType != DataType::f32) throw Error::unsupportedDataTypeCombination(std::string(what) + " must be f32.");
            requireElements(*w, n, what);
        };
        f32vec(a.qNorm, d_.Hd, "DecodeAttention q_norm");
        f32vec(a.kNorm, d_.Hd, "DecodeAttention k_norm");
        f32vec(a.invFreq, d_.Hd / 2, "DecodeAttention inv_freq");
        dc_.flags = (a.qNorm ? 1u : 0u) | (a.kNorm ? 2u : 0u) | (a.vNorm ? 4u : 0u) | (a.invFreq ? 8u : 0u);
        dc_.eps = a.eps;
        dc_.ropeScaling = a.ropeScaling;
        dc_.rowStride = (uint32_t)rowStride;
        const Tensor &dummy = qkv_;  // bound in place of an absent optional input; never read
        wq_ = a.qNorm ? *a.qNorm : dummy;
        wk_ = a.kNorm ? *a.kNorm : dummy;
        invf_ = a.invFreq ? *a.invFreq : dummy;
        mask_ = a.mask;
        scale_ = a.scale;
        const bool alignedOk = aligned16(qkv_.data) && aligned16(k_.data) && aligned16(v_.data) && (rowStride * stride(t)) % 16 == 0;
        plan_ = fdPlan(t, d_, alignedOk, d_.cap);
        if (!plan_.lpk)
            throw Error::unsupportedDataTypeCombination(
                "DecodeAttention needs 16-byte aligned f16/bf16 data with head dim 64, 128, 256 or 512 (f32: 128, 256, 512).");
        partialName_ = std::string("flash_decoding_fresh_") + tag(t) + plan_.suffix();
        reduceName_ = std::string("flash_decoding_reduce_") + tag(out_.dataType) + "_ext";
    }

    std::vector<Binding> tensors() const override {
        return {{qkv_, kRead}, {k_, kReadWrite}, {v_, kReadWrite}, {out_, kWrite}, {pos_, kRead},
                {wq_, kRead}, {wk_, kRead}, {invf_, kRead}};
    }
    std::string describe() const override { return partialName_ + "," + reduceName_; }

    void encode(KernelCommandEncoder &enc) const override {
        const int64_t P = plan_.P;
        const int64_t slots = d_.B * d_.Nq * P;
        enc.withTemporaryTensor(ScratchSpec{{slots, d_.Hd}, DataType::f32}, [&](Tensor pO) {
            enc.withTemporaryTensor(ScratchSpec{{slots}, DataType::f32}, [&](Tensor pM) {
                enc.withTemporaryTensor(ScratchSpec{{slots}, DataType::f32}, [&](Tensor pL) {
                    FlashDecodingPartialExtConstants pc{};
                    pc.B = (uint32_t)d_.B;
                    pc.Nq = (uint32_t)d_.Nq;
                    pc.Nkv = (uint32_t)d_.Nkv;
                    pc.Sk = (uint32_t)d_.cap;
                    pc.Hd = (uint32_t)d_.Hd;
                    pc.P = (uint32_t)P;
                    pc.maskKind = mask_.kind;
                    pc.slidingWindow = mask_.kind == 1 ? mask_.window : -1;
                    pc.scale = scale_;
                    pc.kvStride = (uint32_t)d_.cap;
                    pc.Sq = 1;
                    pc.keyLenFromPosition = 1;
                    DispatchSize ds;
                    ds.grid = dim3((unsigned)P, (unsigned)(d_.B * d_.Nkv * plan_.ngroups), 1);
                    ds.block = dim3((unsigned)plan_.block(), 1, 1);
                    FixedDispatch partial(partialName_,
                                          {{qkv_, kRead}, {k_, kReadWrite}, {v_, kReadWrite}, {pO, kWrite}, {pM, kWrite},
                                           {pL, kWrite}, {pos_, kRead}, {wq_, kRead}, {wk_, kRead}, {invf_, kRead}},
                                          {bytesOf(pc), bytesOf(dc_)}, ds);
                    enc.dispatch(partial);
                    FlashDecodingReduceExtConstants rc{};
                    rc.B = (uint32_t)d_.B;
                    rc.Nq = (uint32_t)d_.Nq;
                    rc.Hd = (uint32_t)d_.Hd;
                    rc.P = (uint32_t)P;
                    rc.Sq = 1;
                    DispatchSize rs;
                    rs.grid = dim3((unsigned)(d_.B * d_.Nq), (unsigned)cdiv(d_.Hd, 64), 1);
                    rs.block = dim3(kBlock, 1, 1);
                    FixedDispatch reduce(reduceName_, {{pO, kRead}, {pM, kRead}, {pL, kRead}, {out_, kWrite}},
                                         {bytesOf(rc)}, rs);
                    enc.dispatch(reduce);
                });
            });
        });
    }

private:
    Tensor qkv_, k_, v_, out_, pos_, wq_, wk_, invf_;
    AttnDims d_{};
    DecodeAttentionConstants dc_{};
    AttentionMask mask_{0, -1};
    float scale_ = 1.0f;
    FdPlan plan_;
    std::string partialName_, reduceName_;
};

// ---------------------------------------------------------------------------
// Matmul (Matmul.swift)
// ---------------------------------------------------------------------------

// The streaming matvec for a transposeB product with m == 1 (the triples of
// Matmul.swift:362-374, plus f16 triples): matvec_nk_stream_<x>_<w>_<o>,
// suffixed _r<R> by the caller.
std::string matvecNKName(DataType x, DataType w, DataType o) {
    using D = DataType;
    const bool ok = (x == D::f32 && w == D::f32 && o == D::f32) || (x == D::f32 && w == D::bf16 && o == D::f32) ||
                    (x == D::bf16 && w == D::bf16 && o == D::f32) || (x == D::bf16 && w == D::bf16 && o == D::bf16) ||
                    (x == D::f32 && w == D::f16 && o == D::f32) || (x == D::f16 && w == D::f16 && o == D::f32) ||
                    (x == D::f16 && w == D::f16 && o == D::f16);
    if (!ok) return "";
    return std::string("matvec_nk_stream_") + tag(x) + "_" + tag(w) + "_" + tag(o);
}

std::string plainName(const char *base, DataType x, DataType w, DataType o) {
    using D = DataType;
    std::string b = base;
    // Matmul.swift:222-229 and :381-388, plus f16 triples
    if (x == D::f32 && w == D::f32 && o == D::f32) return b;
    if (x == D::f32 && w == D::f16 && o == D::f32) return b + "_f16";
    if (x == D::f32 && w == D::bf16 && o == D::f32) return b + "_bf16";
    if (x == D::bf16 && w == D::bf16 && o == D::f32) return b + "_bf16_bf16_f32";
    if (x == D::bf16 && w == D::bf16 && o == D::bf16) return b + "_bf16_bf16_bf16";
    if (x == D::f16 && w == D::f16 && o == D::f32) return b + "_f16_f16_f32";
    if (x == D::f16 && w == D::f16 && o == D::f16) return b + "_f16_f16_f16";
    return "";
}

// Rows per unit of the streaming matvecs (stream.hpp): 4 for long outputs
// (one LDS read of x feeds 4 rows), 1 otherwise (finer units balance better).
int matvecRows(int64_t N) { return N >= 32768 ? 4 : 1; }

// Waves per CU the streaming kernels are sized for: 12 (3 blocks of 4 waves,
// 3 waves per SIMD), measured best on MI355X for the decode matvecs with 4
// steps in flight per wave (stream.hpp); POPCORN_STREAM_WAVES_PER_CU
// overrides it (1..32) for tuning.
int streamWavesPerCU() {
    static const int w = [] {
        const char *e = std::getenv("POPCORN_STREAM_WAVES_PER_CU");
        const int v = e ? std::atoi(e) : 0;
        return v >= 1 && v <= 32 ? v : 12;
    }();
    return w;
}

// Blocks (of 4 waves) for `units` units: each wave's share is
// ceil(units / maxWaves), and just enough waves are launched to cover the
// units at that share, so every wave streams the same number of units give
// or take one.
int64_t streamBlocks(int64_t units) {
    if (units <= 0) return 0;
    const int64_t maxWaves = (int64_t)deviceCUs() * streamWavesPerCU();
    const int64_t per = cdiv(units, maxWaves);
    return cdiv(cdiv(units, per), kBlock / 64);
}

// The 4-bit fast kernels' launch shape: lanes per row LPR (8, 12, 16 or 32;
// a unit is floor(64 / LPR) rows and a row's K / 64 groups are dealt to its
// LPR lanes, one group per lane and step) and x octets per thread J (2 or
// 8). LPR minimises the steps of the busiest SIMD, waves per SIMD x units
// per wave x steps per unit, at the grid's waves per CU (the 4-bit inner
// loop is bound by its vector ALU work): short matrices want many small
// units, long ones full lanes (12 lanes fit rows of 36 groups, K 2304, in 3
// whole steps, where 16 lanes take 3 steps with a quarter of them idle).
// Ties go to the higher lane occupancy.
struct Q4Shape {
    int lpr = 0, j = 0;
};

Q4Shape q4Shape(int64_t N, int64_t K, bool xF32) {
    Q4Shape q;
    const int64_t G = K / 64;
    const int64_t kMax = xF32 ? 4096 : 16384;
    // the fast kernels read a row's scales and biases as 32-bit words, and
    // the packed words through 32-bit byte offsets
    if (N <= 0 || G <= 0 || G % 2 != 0 || K > kMax || N * (K / 2) >= (int64_t{1} << 31)) return q;
    q.j = K <= 4096 ? 2 : 8;
    const int64_t waves = (int64_t)deviceCUs() * streamWavesPerCU();
    int64_t bestSteps = INT64_MAX;
    double bestEff = 0.0;
    const int64_t simds = (int64_t)deviceCUs() * 4;
    for (int lpr : {32, 16, 12, 8}) {
        const int64_t cpl = cdiv(G, lpr), rows = 64 / lpr, units = cdiv(N, rows);
        const int64_t used = std::min(units, waves);
        const int64_t steps = cdiv(used, simds) * cdiv(units, used) * cpl;
        const double eff = (double)G / (double)(lpr * cpl) * (double)(rows * lpr) / 64.0;
        if (steps < bestSteps || (steps == bestSteps && eff > bestEff)) {
            bestSteps = steps;
            bestEff = eff;
            q.lpr = lpr;
        }
    }
    return q;
}

// MFMA GEMM tile shapes (gemm_mfma.hip): BM x BN and the block size.
struct GemmTile {
    int bm, bn, threads;
    const char *suffix;
};

// "e" and "f" tiles copy whole 128-byte lines global -> LDS (stages of K 64,
// the last one's chunks past K reading zeros; 2 stages, or 4 in the "f"
// forms, by buffer loads whose byte offsets stay below 2^31 over a tile's
// rows). "d" tiles copy 64-byte rows (4 stages of K 32) and keep K % 64 ==
// 32, which they fill in whole stages.
bool gemmOffsetsFit(int64_t k, int bn) { return (int64_t)(bn + 16) * k * 2 < (int64_t{1} << 31); }
bool gemmLinesFit(int64_t k, int bn) { return k % 64 != 32 && gemmOffsetsFit(k, bn); }

// The whole-line tiles are chosen by a score: the share of the CU slots
// their grid keeps busy over its rounds (two blocks per CU for the tiles
// of at most 80 KB of LDS; such a tile alone on a CU counts 0.6 of a
// slot), times the share of the grid's tiles that lies inside C, times the
// tile's throughput per CU relative to 256 x 384 when the CUs are full.
// A first round that gives only some CUs their second block is paid in full
// by those: 0.78, measured at M > 512 and K <= 4096 (M 1000, K 2304, N 9216,
// 384 tiles of 128 x 192: 53.4 us, 192 of 256 x 192: 45.0); with fewer rows
// or longer K the larger tiles gave nothing (M 594, K 9216, N 14336: 187
// and 197).
// The weights are fitted to every tile's time on 131 shapes (bf16, M 65-4700,
// K 1024-14336, N 2304-256000, more than two 128 x 128 tiles per CU): the
// score's pick is on average 0.6% slower than the fastest tile (the six tiles
// before 192 x 384, 192 x 256, 256 x 192 and 256 x 320 came in, at their older
// weights: 4.1%), none over 1% slower than those six's pick and the best 1.29
// times as fast (M 1105, K 3072, N 28672: 231 -> 185 us; M 700, K 3072, N
// 24576: 116 -> 98).
struct ScoredTile {
    GemmTile tile;
    int blocksPerCU;
    double weight;
};
const ScoredTile kLineTiles[] = {
    {{256, 384, 512, "e256x384"}, 1, 1.0},  {{256, 320, 512, "e256x320"}, 1, 0.98}, {{192, 384, 768, "e192x384"}, 1, 0.92},
    {{256, 256, 512, "e256x256"}, 1, 0.90}, {{256, 288, 768, "e256x288"}, 1, 0.93}, {{128, 192, 256, "e128x192"}, 2, 0.81},
    {{256, 192, 512, "e256x192"}, 1, 0.80}, {{192, 256, 768, "e192x256"}, 1, 0.74}, {{128, 128, 256, "e128x128"}, 2, 0.72}};

double lineTileScore(const ScoredTile &t, int64_t m, int64_t n, int64_t k) {
    const int64_t cus = deviceCUs();
    const int64_t tm = cdiv(m, t.tile.bm), tn = cdiv(n, t.tile.bn), tiles = tm * tn;
    const int64_t slots = cus * t.blocksPerCU;
    double fill = (double)tiles / (double)(cdiv(tiles, slots) * slots);
    if (t.blocksPerCU > 1 && tiles <= cus) fill = 0.6 * (double)tiles / (double)cus;
    else if (t.blocksPerCU > 1 && tiles < slots && m > 512 && k <= 4096) fill *= 0.78;
    const double inside = (double)(m * n) / (double)(tm * t.tile.bm * tn * t.tile.bn);
    return fill * inside * t.weight;
}

const ScoredTile &bestLineTile(int64_t m, int64_t n, int64_t k) {
    const ScoredTile *best = &kLineTiles[0];
    double bestScore = -1.0;
    for (const ScoredTile &t : kLineTiles) {
        const double sc = lineTileScore(t, m, n, k);
        if (sc > bestScore) {
            bestScore = sc;
            best = &t;
        }
    }
    return *best;
}

// Small grids: products of at least 2^29 multiply-adds (below that a product
// is mostly launch and one 128 x 128 pass keeps it at one launch) whose
// 128 x 128 tiles give no more than two per CU. There the CUs, not the tile's
// rate, set the time, so the plan chooses a tile and a number of K splits
// together, by the time that a block's stages take:
//   rounds of blocks x (stages per block x us per stage + us per block)
//   + for a split, the reduction's launch and its partials' trip through HBM,
// with us per stage from a fit over 68 shapes (bf16, m 65-1800, the
// projections of the Gemma shapes and odd sizes, 1 to 16 splits; the plan's
// pick is on average 2% slower than the fastest of every tile and split, 20%
// at worst). M 137, K 9216, N 2304: 85.9 us on 36 tiles of 128 x 128, 19.8
// on 128 x 128 tiles and 7 splits; M 1000, K 9216, N 2304: 91.5 -> 51; M 1000,
// K 2304, N 1024: 25.6 -> 13.3 on 64 x 64 tiles. With more than two tiles per
// CU the score above is as good (M 1000, K 2304, N 9216: 48.8 both ways).
struct SmallTile {
    GemmTile tile;
    int blocksPerCU;
    double alone, full, block;  // us per stage with one block per CU, with the CU full, and us per block
};
const SmallTile kSmallTiles[] = {{{64, 64, 256, "f64x64"}, 2, 0.313, 0.500, 0.2},
                                 {{128, 64, 256, "f128x64"}, 1, 0.402, 0.407, 0.8},
                                 {{128, 128, 256, "e128x128"}, 2, 0.790, 1.209, 0.6},
                                 {{128, 128, 256, "f128x128"}, 1, 0.604, 0.662, 1.6},
                                 {{256, 256, 512, "e256x256"}, 1, 1.620, 1.932, 0.4}};
constexpr int kE128 = 2;

bool gemmSmallGrid(int64_t m, int64_t n, int64_t k) {
    return (double)m * (double)n * (double)k >= 0x1p29 && cdiv(m, 128) * cdiv(n, 128) <= 2 * (int64_t)deviceCUs() &&
           gemmOffsetsFit(k, 384);
}

struct GemmPlan {
    GemmTile tile;
    int64_t splits;
};

GemmPlan gemmSmallPlan(int64_t m, int64_t n, int64_t k, bool maySplit) {
    const int64_t cus = deviceCUs(), stages = cdiv(k, 64);
    GemmPlan best{kSmallTiles[0].tile, 1};
    double bestUs = 1e30, unsplit128 = 0.0;
    for (const SmallTile &t : kSmallTiles) {
        const int64_t tiles = cdiv(m, t.tile.bm) * cdiv(n, t.tile.bn);
        // a split takes at least 4 stages; more than 16 were never the fastest
        for (int64_t s = 1; s <= 16 && (s == 1 || (maySplit && stages / s >= 4)); ++s) {
            const int64_t slots = cus * t.blocksPerCU, rounds = tiles * s / slots, rest = tiles * s % slots;
            const double per = (double)cdiv(stages, s), over = std::max(0.0, (double)rest / (double)cus - 1.0);
            double us = (double)rounds * (per * t.full + t.block);
            if (rest) us += per * (t.alone + (t.full - t.alone) * over) + t.block;
            if (s > 1) us += 4.3 + 0.14 * 8e-6 * (double)s * (double)m * (double)n;
            if (s == 1 && &t == &kSmallTiles[kE128]) unsplit128 = us;
            if (us < bestUs) {
                bestUs = us;
                best = GemmPlan{t.tile, s};
            }
        }
    }
    // 128 x 128 tiles of whole stages on more than one but not two full rounds
    // of the CUs run up to 30% faster than their estimate (which is near on fewer
    // tiles), so splits of 256 x 256 must beat it by more there: M 389, K 4096, N
    // 14336, bf16: 50.9 us, split 60.4; M 1156, K 4096, N 4096 46.4 and 52.5; but
    // M 1015, K 14336, N 4096 152 and 115 (300 shapes: with 0.85 none is over 4%
    // slower than unsplit, 3 give up 3 to 17%).
    const int64_t tiles = cdiv(m, 128) * cdiv(n, 128);
    if (best.splits > 1 && best.tile.bm == 256 && k % 64 == 0 && tiles > cus && bestUs > 0.85 * unsplit128)
        best = GemmPlan{kSmallTiles[kE128].tile, 1};
    return best;
}

GemmTile gemmTileForm(int64_t m, int64_t n, int64_t k);
GemmTile gemmTile(int64_t m, int64_t n, int64_t k) {
    if (!std::getenv("POPCORN_GEMM_TILE") && gemmLinesFit(k, 384)) return bestLineTile(m, n, k).tile;
    return gemmTileForm(m, n, k);
}

GemmTile gemmTileForm(int64_t m, int64_t n, int64_t k) {
    static const GemmTile tiles[] = {{256, 256, 512, "d256x256"}, {128, 128, 256, "d128x128"},
                                     {128, 256, 512, "d128x256"}, {128, 192, 256, "d128x192"},
                                     {256, 384, 512, "d256x384"}, {256, 256, 512, "e256x256"},
                                     {128, 128, 256, "e128x128"}, {128, 256, 512, "e128x256"},
                                     {128, 192, 256, "e128x192"}, {256, 384, 512, "e256x384"},
                                     {256, 288, 768, "e256x288"}, {64, 64, 256, "f64x64"},
                                     {128, 64, 256, "f128x64"},   {128, 128, 256, "f128x128"},
                                     {256, 320, 512, "e256x320"}, {192, 384, 768, "e192x384"},
                                     {256, 192, 512, "e256x192"}, {192, 256, 768, "e192x256"}};
    if (const char *e = std::getenv("POPCORN_GEMM_TILE")) {  // tuning override, e.g. "e128x192"
        for (const GemmTile &t : tiles)
            if (std::string(t.suffix) == e && (t.suffix[0] == 'd' ? k % 32 == 0 : gemmOffsetsFit(k, std::max(t.bm, t.bn)))) return t;
    }
    if (k % 32 != 0) return tiles[6];  // an override that does not fit
    // 256 x 256 on 8 waves reuses each LDS stage for twice the MFMA work of
    // 128 x 128 but runs one block per CU, so it only pays when the tiles
    // fill the CUs several times over; below that the 128 x 128 grid (two
    // blocks per CU) balances better (config 5, f16, M 2048; us):
    //                      d256  d128
    //   QKV  N 9216  K 3072   177   162
    //   gate N 24576 K 3072   319   422
    //   down N 3072  K 24576  589   430
    // 256 x 384 (8 waves of 128 x 96: 7 fragment reads per 12 MFMAs) when
    // its grid keeps at least 70% of the CUs busy in every round
    // (config-5 QKV, 192 tiles: 136 -> 127 us; gate and up, 512 tiles:
    // 294-303 -> 284-288 us)
    const int64_t cus = deviceCUs();
    const int64_t t384 = cdiv(m, 256) * cdiv(n, 384);
    if (t384 * 10 >= cus * 7 && t384 * 10 >= cdiv(t384, cus) * cus * 7) return tiles[4];
    if (cdiv(m, 256) * cdiv(n, 256) >= 3 * cus) return tiles[0];
    // 128 x 192 tiles when their grid is whole rounds of one tile per CU
    // (config-5 QKV, N 9216: 768 tiles, 155 -> 135 us; down, N 3072:
    // 256 tiles, 397 -> 352 us)
    const int64_t t192 = cdiv(m, 128) * cdiv(n, 192);
    if (n % 192 == 0 && t192 % cus == 0) return tiles[3];
    // a 128 x 128 grid between one and two tiles per CU leaves half the
    // CUs with a second tile; one 128 x 256 tile per CU (8 waves) ends
    // sooner (config-5 down: 379 against 423 us before 128 x 192 took it)
    const int64_t t128 = cdiv(m, 128) * cdiv(n, 128);
    if (t128 > cus && t128 < 2 * cus && n >= 256) return tiles[2];
    return tiles[1];
}

// Split-K for a GEMM whose 256 x 384 tiles are too few to fill the CUs:
// the number of K splits that makes the grid whole rounds of one tile per
// CU, each split at least 2048 deep, or 0. Config-5 down (M 2048, N 3072,
// K 24576): 64 tiles x 4 splits of K 6144.
int64_t gemmSplitK(int64_t m, int64_t n, int64_t k) {
    if (std::getenv("POPCORN_GEMM_TILE") || k % 32 != 0 || (m * n) % 4 != 0) return 0;
    const int64_t cus = deviceCUs();
    const int64_t t384 = cdiv(m, 256) * cdiv(n, 384);
    if (t384 * 10 >= cus * 7) return 0;
    for (int64_t s = 2; s <= 8; ++s)
        if ((t384 * s) % cus == 0 && k % (32 * s) == 0 && k / s >= 2048) {
            // with whole-line tiles, split only when it beats the best tile's
            // score: the split grid fills the CUs, less its tiles' share
            // outside C and the share of time that its partials' round trip
            // through HBM adds (8 s bytes per element at ~7 TB/s against 2 K
            // flop at ~1.2 PFLOP/s: ~700 s / K). 1.1: the scores rank tiles
            // over all fills, and a nearly full grid does better than its
            // score says (f16, unsplit and split: M 2048, N 6144, K 8192: 185
            // and 205 us, K 14336: 345 and 322; M 512, N 12288, K 8192: 140
            // and 121; M 375, N 24576, K 4096: 100 and 112)
            if (gemmLinesFit(k, 384)) {
                const ScoredTile &t = bestLineTile(m, n, k);
                const double inside = (double)(m * n) / (double)(t384 * 256 * 384);
                if (inside * (1.0 - 700.0 * (double)s / (double)k) <= 1.1 * lineTileScore(t, m, n, k)) return 0;
            }
            return s;
        }
    return 0;
}

// The split-K GEMM: f32 partial products per split in scratch, then one
// pass that sums them and rounds to C's dtype. Without scratch the whole
// product runs on unsplit tiles.
class SplitKMatmulKernel : public Kernel {
public:
    SplitKMatmulKernel(const Tensor &a, const Tensor &b, const Tensor &c, int64_t m, int64_t k, int64_t n, GemmPlan plan)
        : a_(a), b_(b), c_(c), m_(m), k_(k), n_(n), splits_(plan.splits), tile_(plan.tile) {}
    std::vector<Binding> tensors() const override { return {{a_, kRead}, {b_, kRead}, {c_, kWrite}}; }
    std::string describe() const override { return mainName() + "," + reduceName(); }
    void encode(KernelCommandEncoder &enc) const override {
        MatmulConstants mc{(uint32_t)m_, (uint32_t)k_, (uint32_t)n_, 1u};
        const bool done = enc.tryTemporaryTensor(ScratchSpec{{splits_ * m_, n_}, DataType::f32}, [&](Tensor part) {
            DispatchSize ds;
            ds.grid = dim3((unsigned)(cdiv(m_, tile_.bm) * cdiv(n_, tile_.bn)), (unsigned)splits_, 1);
            ds.block = dim3((unsigned)tile_.threads, 1, 1);
            FixedDispatch s1(mainName(), {{a_, kRead}, {b_, kRead}, {part, kWrite}}, {bytesOf(mc)}, ds);
            enc.dispatch(s1);
            const uint32_t splits = (uint32_t)splits_;
            const int64_t blocks = std::clamp<int64_t>(cdiv(m_ * n_ / 4, kBlock), 1, 8 * deviceCUs());
            FixedDispatch s2(reduceName(), {{part, kRead}, {c_, kWrite}}, {bytesOf(mc), bytesOf(splits)}, grid1(blocks, kBlock));
            enc.dispatch(s2);
        });
        if (done) return;
        const GemmTile tile = gemmTile(m_, n_, k_);
        FixedDispatch whole(std::string("matmul_mfma_") + tag(a_.dataType) + "_" + tag(a_.dataType) + "_" +
                                tag(c_.dataType) + "_" + tile.suffix,
                            {{a_, kRead}, {b_, kRead}, {c_, kWrite}}, {bytesOf(mc)},
                            grid1(cdiv(m_, tile.bm) * cdiv(n_, tile.bn), tile.threads));
        enc.dispatch(whole);
    }

private:
    std::string mainName() const { return std::string("matmul_mfma_") + tag(a_.dataType) + "_splitk_" + tile_.suffix; }
    std::string reduceName() const { return std::string("matmul_splitk_reduce_") + tag(c_.dataType); }
    Tensor a_, b_, c_;
    int64_t m_, k_, n_, splits_;
    GemmTile tile_;
};

constexpr int64_t kMaxStagedK = 16384;  // x staged as f32 in 64 KB of LDS
// A Matmul with a non-transposed 16-bit B [K, N] and m > 1: B^T into
// scratch (transpose2d_b16), then the transposed-B route (the MFMA or
// skinny kernels) on it.
std::unique_ptr<Kernel> makeMatmul(const Tensor &a, const Tensor &b, const Tensor &c, int64_t m, int64_t k, int64_t n,
                                   bool transposeB);
class TransposeBMatmulKernel : public Kernel {
public:
    TransposeBMatmulKernel(const Tensor &a, const Tensor &b, const Tensor &c, int64_t m, int64_t k, int64_t n)
        : a_(a), b_(b), c_(c), m_(m), k_(k), n_(n) {}
    std::vector<Binding> tensors() const override { return {{a_, kRead}, {b_, kRead}, {c_, kWrite}}; }
    std::string describe() const override {
        // the inner route's kernels, for B^T in (256-byte aligned) scratch
        Tensor bt(reinterpret_cast<void *>(uintptr_t{1} << 20), Shape({n_, k_}), b_.dataType);
        return "transpose2d_b16," + makeMatmul(a_, bt, c_, m_, k_, n_, true)->describe();
    }
    void encode(KernelCommandEncoder &enc) const override {
        enc.withTemporaryTensor(ScratchSpec{{n_, k_}, b_.dataType}, [&](Tensor bt) {
            Transpose2DConstants tc{(uint32_t)k_, (uint32_t)n_};
            DispatchSize ds;
            ds.grid = dim3((unsigned)cdiv(n_, 64), (unsigned)cdiv(k_, 64), 1);
            ds.block = dim3(kBlock, 1, 1);
            FixedDispatch t("transpose2d_b16", {{b_, kRead}, {bt, kWrite}}, {bytesOf(tc)}, ds);
            enc.dispatch(t);
            makeMatmul(a_, bt, c_, m_, k_, n_, true)->encode(enc);
        });
    }

private:
    Tensor a_, b_, c_;
    int64_t m_, k_, n_;
};


std::unique_ptr<Kernel> makeMatmul(const Tensor &a, const Tensor &b, const Tensor &c, int64_t m, int64_t k, int64_t n,
                                   bool transposeB) {
    if (m < 0 || k < 0 || n < 0) throw Error::tensorShapeMismatch("Matmul dimensions must be non-negative.");
    requireElements(a, m * k, "Matmul a");
    requireElements(b, k * n, "Matmul b");
    requireElements(c, m * n, "Matmul c");
    std::vector<Binding> binds = {{a, kRead}, {b, kRead}, {c, kWrite}};
    if (m == 1) {
        // Matmul.swift:233-277
        MatvecConstants mc{(uint32_t)k, (uint32_t)n, transposeB ? 1u : 0u};
        if (transposeB) {
            std::string fn = matvecNKName(a.dataType, b.dataType, c.dataType);
            if (fn.empty())
                throw Error::unsupportedDataTypeCombination(std::string("Unsupported matvec data type combination: ") +
                                                            tag(a.dataType) + ", " + tag(b.dataType) + ", " + tag(c.dataType) + ".");
            if (k > kMaxStagedK) throw Error::tensorShapeMismatch("matvec K above " + std::to_string(kMaxStagedK) + " is not supported.");
            const int R = matvecRows(n);
            fn += "_r" + std::to_string(R);
            return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)},
                                                   grid1(streamBlocks(cdiv(n, R)), kBlock, (size_t)std::max<int64_t>(k, 1) * 4));
        }
        std::string fn = plainName("matvec", a.dataType, b.dataType, c.dataType);
        if (fn.empty())
            throw Error::unsupportedDataTypeCombination(std::string("Unsupported matvec data type combination: ") +
                                                        tag(a.dataType) + ", " + tag(b.dataType) + ", " + tag(c.dataType) + ".");
        return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)}, grid1(cdiv(n, kBlock), kBlock));
    }
    // m > 1, transposeB, 16-bit operands: the MFMA tiles (the reference's MPP
    // GEMM path, Matmul.swift:175-196); 16-byte rows needed (K % 8 == 0).
    {
        const DataType t = a.dataType;
        // a [K, N] B (the reference's mpp_matmul without _tb): transposed
        // into scratch first, then this route (the scratch is 256-byte aligned)
        if (!transposeB && (t == DataType::f16 || t == DataType::bf16) && b.dataType == t &&
            (c.dataType == t || c.dataType == DataType::f32) && k % 8 == 0 && k > 0 && aligned16(a.data) &&
            k < 65536 * 64 && n < 65536 * 64)
            return std::make_unique<TransposeBMatmulKernel>(a, b, c, m, k, n);
        if (transposeB && (t == DataType::f16 || t == DataType::bf16) && b.dataType == t &&
            (c.dataType == t || c.dataType == DataType::f32) && k % 8 == 0 && k > 0 && aligned16(a.data) &&
            aligned16(b.data)) {
            // 2 <= M <= 64: the skinny kernel (gemm_skinny.hip), which
            // streams B once with its K split over a block's waves: about
            // 3 waves per CU in all, at most 4 per block (measured best on
            // MI355X for N 2304..24576 x K 2304..9216)
            if (m <= 64 && !std::getenv("POPCORN_GEMM_TILE") && n * k * 2 <= INT32_MAX && m * k * 2 <= INT32_MAX) {
                const int mt = (int)cdiv(m, 16);
                MatmulConstants mc{(uint32_t)m, (uint32_t)k, (uint32_t)n, 1u};
                // at least 512 tiles of 16 rows of B: A staged in LDS, one
                // tile per wave (one wave per block at M <= 16, else four)
                if (cdiv(n, 16) >= 2 * (int64_t)deviceCUs()) {
                    const int w = mt == 1 ? 1 : 4;
                    const std::string fn = std::string("matmul_skinny_") + tag(t) + "_" + tag(t) + "_" + tag(c.dataType) +
                                           "_m" + std::to_string(16 * mt) + "_lds";
                    return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)},
                                                           grid1(cdiv(cdiv(n, 16), w), 64 * w));
                }
                // 16-row blocks (_r16) when 32-row ones would be fewer than the CUs
                const int rows = cdiv(n, 32) < deviceCUs() ? 16 : 32;
                const int64_t blocks = cdiv(n, rows);
                const int64_t want = 3 * (int64_t)deviceCUs() / blocks;
                int64_t w = 1;
                while (2 * w <= want && w < 4 && 2 * w <= cdiv(k, 32)) w *= 2;
                const std::string fn = std::string("matmul_skinny_") + tag(t) + "_" + tag(t) + "_" + tag(c.dataType) +
                                       "_m" + std::to_string(16 * mt) + (rows == 16 ? "_r16" : "");
                return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)},
                                                       grid1(blocks, (int)(64 * w)));
            }
            // (rows too long for 32-bit offsets over a tile that the 64-byte-row
            // tiles do not take either go to the SIMT tiles below)
            if (k % 32 == 0 || gemmOffsetsFit(k, 384)) {
                // the split-K reduction stores 4 results of C at a time
                if (const int64_t splits = aligned16(c.data) ? gemmSplitK(m, n, k) : 0) {
                    // each split's K a whole number of 64-deep stages
                    const bool lines = gemmLinesFit(k, 384) && k % (64 * splits) == 0;
                    return std::make_unique<SplitKMatmulKernel>(
                        a, b, c, m, k, n, GemmPlan{{256, 384, 512, lines ? "e256x384" : "d256x384"}, splits});
                }
                MatmulConstants mc{(uint32_t)m, (uint32_t)k, (uint32_t)n, 1u};
                GemmTile tile = gemmTile(m, n, k);
                if (!std::getenv("POPCORN_GEMM_TILE") && gemmSmallGrid(m, n, k)) {
                    const GemmPlan plan = gemmSmallPlan(m, n, k, aligned16(c.data));
                    if (plan.splits > 1) return std::make_unique<SplitKMatmulKernel>(a, b, c, m, k, n, plan);
                    tile = plan.tile;
                }
                const std::string fn =
                    std::string("matmul_mfma_") + tag(t) + "_" + tag(t) + "_" + tag(c.dataType) + "_" + tile.suffix;
                return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)},
                                                       grid1(cdiv(m, tile.bm) * cdiv(n, tile.bn), tile.threads));
            }
        }
    }
    // m > 1 with f32 output and an f32 operand (the reference's MPP f32
    // combinations f32 x f32, f32 x bf16, bf16 x f32, Matmul.swift:203-214):
    // the f32 matrix-core tiles (gemm_f32.hip), B either way round; rows of
    // 4 values in 16-byte-aligned buffers
    {
        const DataType ta = a.dataType, tb = b.dataType, f32 = DataType::f32, bf16 = DataType::bf16;
        const bool combo = c.dataType == f32 && ((ta == f32 && (tb == f32 || tb == bf16)) || (ta == bf16 && tb == f32));
        if (combo && m > 1 && k % 4 == 0 && (transposeB || n % 4 == 0) && aligned16(a.data) && aligned16(b.data)) {
            MatmulConstants mc{(uint32_t)m, (uint32_t)k, (uint32_t)n, transposeB ? 1u : 0u};
            const std::string fn = std::string("matmul_mfma_") + tag(ta) + "_" + tag(tb) + "_f32" + (transposeB ? "_tb" : "");
            return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)},
                                                   grid1(cdiv(m, 128) * cdiv(n, 128), kBlock));
        }
    }
    // the SIMT tiles (matmul.hip) in the place of the reference's matmul_typed
    std::string fn = plainName("matmul_tiled", a.dataType, b.dataType, c.dataType);
    if (fn.empty())
        throw Error::unsupportedDataTypeCombination(std::string("Unsupported matmul data type combination: ") +
                                                    tag(a.dataType) + ", " + tag(b.dataType) + ", " + tag(c.dataType) + ".");
    MatmulConstants mc{(uint32_t)m, (uint32_t)k, (uint32_t)n, transposeB ? 1u : 0u};
    DispatchSize ds;
    ds.grid = dim3((unsigned)cdiv(n, 64), (unsigned)cdiv(m, 64), 1);
    ds.block = dim3(kBlock, 1, 1);
    return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(mc)}, ds);
}

// ---------------------------------------------------------------------------
// Gated MLP (Gemma4TextInference.swift:416-429 as two dispatches)
// ---------------------------------------------------------------------------

class GatedMLPKernel : public Kernel {
public:
    GatedMLPKernel(const Tensor &x, const Tensor *nw, const Tensor &wg, const Tensor &wu, const Tensor &wd, const Tensor &out,
                   float eps, bool addOne, const Tensor *hidden)
        : x_(x), wg_(wg), wu_(wu), wd_(wd), out_(out), eps_(eps), addOne_(addOne) {
        if (nw) {
            nw_ = *nw;
            hasNorm_ = true;
        }
        if (hidden) {
            h_ = *hidden;
            hasHidden_ = true;
        }
        if (wg.shape.rank() != 2) throw Error::tensorInvalidRank(2, wg.shape.rank());
        F_ = wg.shape[0];
        H_ = wg.shape[1];
        if (wu.shape != wg.shape) throw Error::tensorShapeMismatch("GatedMLP up weight shape must match gate weight " + wg.shape.str() + ".");
        if (wd.shape != Shape({H_, F_})) throw Error::tensorShapeMismatch("GatedMLP down weight must be [" + std::to_string(H_) + ", " + std::to_string(F_) + "].");
        if (x.shape.rank() < 1 || x.shape.dims.back() != H_ || x.shape.elementCount() != H_)
            throw Error::tensorShapeMismatch("GatedMLP decodes one row: x must hold [" + std::to_string(H_) + "].");
        if (out.shape != x.shape) throw Error::tensorShapeMismatch("GatedMLP output shape must match x.");
        const DataType t = x.dataType;
        if (!isFloat(t) || wg.dataType != t || wu.dataType != t || wd.dataType != t || out.dataType != t)
            throw Error::unsupportedDataTypeCombination("GatedMLP needs x, weights and out of one float dtype.");
        if (hasNorm_) {
            if (nw_.dataType != DataType::f32) throw Error::unsupportedDataTypeCombination("GatedMLP norm weight must be f32.");
            requireElements(nw_, H_, "GatedMLP norm weight");
        }
        if (hasHidden_) {
            if (h_.dataType != t) throw Error::unsupportedDataTypeCombination("GatedMLP hidden must have x's dtype.");
            requireElements(h_, F_, "GatedMLP hidden");
        }
        if (H_ > kMaxStagedK || F_ > kMaxStagedK) throw Error::tensorShapeMismatch("GatedMLP H and F must be <= 16384.");
        requireElements(x, H_, "x");
        requireElements(wg, F_ * H_, "w_gate");
        requireElements(wu, F_ * H_, "w_up");
        requireElements(wd, H_ * F_, "w_down");
        R_ = F_ >= 32768 ? 2 : 1;
        down_ = makeMatmul(wd_, wd_, out_, 1, F_, H_, true);  // name/geometry probe only
    }

    // Residual form: x_ is the incoming residual stream; x = x_ +
    // RMSNorm(delta) * wPost is stored to xOut and feeds the MLP.
    void setResidual(const Tensor &delta, const Tensor &wPost, const Tensor &xOut) {
        if (delta.dataType != x_.dataType || xOut.dataType != x_.dataType)
            throw Error::unsupportedDataTypeCombination("GatedMLP residual tensors must have x's dtype.");
        if (wPost.dataType != DataType::f32) throw Error::unsupportedDataTypeCombination("post-norm weight must be f32.");
        requireElements(delta, H_, "GatedMLP delta");
        requireElements(wPost, H_, "GatedMLP post-norm weight");
        requireElements(xOut, H_, "GatedMLP x_out");
        if (xOut.data == x_.data) throw Error::invalidArgument("GatedMLP x_out must not alias x (blocks read x while block 0 writes x_out)");
        delta_ = delta;
        wPost_ = wPost;
        xOut_ = xOut;
        residual_ = true;
    }

    std::vector<Binding> tensors() const override {
        std::vector<Binding> b = {{x_, kRead}, {wg_, kRead}, {wu_, kRead}, {wd_, kRead}, {out_, kWrite}};
        if (hasNorm_) b.push_back({nw_, kRead});
        if (hasHidden_) b.push_back({h_, kWrite});
        if (residual_) {
            b.push_back({delta_, kRead});
            b.push_back({wPost_, kRead});
            b.push_back({xOut_, kWrite});
        }
        return b;
    }

    std::string describe() const override { return gateUpName() + "," + down_->describe(); }

    std::string gateUpName() const {
        return std::string("gated_mlp_gate_up_") + tag(x_.dataType) + (R_ == 1 ? "_r1" : "") + (residual_ ? "_res" : "");
    }

    void encode(KernelCommandEncoder &enc) const override {
        auto run = [&](const Tensor &h) {
            GatedMLPConstants gc{(uint32_t)H_, (uint32_t)F_, hasNorm_ ? 1u : 0u, addOne_ ? 1u : 0u, eps_,
                                 (uint32_t)x_.dataType, residual_ ? 1u : 0u};
            const Tensor normOrDummy = hasNorm_ ? nw_ : x_;
            // delta, w_post and x_out are touched only in the residual form
            const Tensor d = residual_ ? delta_ : x_, w = residual_ ? wPost_ : x_, xo = residual_ ? xOut_ : x_;
            FixedDispatch gu(gateUpName(),
                             {{x_, kRead}, {normOrDummy, kRead}, {wg_, kRead}, {wu_, kRead}, {h, kWrite}, {d, kRead},
                              {w, kRead}, {xo, residual_ ? kWrite : kRead}},
                             {bytesOf(gc)}, grid1(streamBlocks(cdiv(F_, R_)), kBlock, (size_t)H_ * 4));
            enc.dispatch(gu);
            auto down = makeMatmul(h, wd_, out_, 1, F_, H_, true);
            down->encode(enc);
        };
        if (hasHidden_) {
            run(h_);
        } else {
            enc.withTemporaryTensor(ScratchSpec{{F_}, x_.dataType}, [&](Tensor h) { run(h); });
        }
    }

private:
    Tensor x_, nw_, wg_, wu_, wd_, out_, h_, delta_, wPost_, xOut_;
    float eps_;
    bool addOne_, hasNorm_ = false, hasHidden_ = false, residual_ = false;
    int64_t H_ = 0, F_ = 0, R_ = 2;
    std::unique_ptr<Kernel> down_;
};

// The gated MLP with block-affine 4-bit gate, up and down weights: the fused
// front half (q4_gate_up_*) then the 4-bit down matvec (aq_qmv_fast_*).
// bf16 activations; the post-attention residual in front when delta is given.
class GatedMLPQ4Kernel : public Kernel {
public:
    GatedMLPQ4Kernel(const Tensor &x, const Tensor &nw, const AffineQuantizedTensor &wg, const AffineQuantizedTensor &wu,
                     const AffineQuantizedTensor &wd, const Tensor &out, float eps, const Tensor *hidden)
        : x_(x), nw_(nw), wg_(wg), wu_(wu), wd_(wd), out_(out), eps_(eps) {
        for (const AffineQuantizedTensor *q : {&wg, &wu, &wd}) {
            q->validate();
            if (q->bits != 4 || q->groupSize != 64 || q->scales.dataType != DataType::bf16 || q->shape.rank() != 2)
                throw Error::unsupportedDataTypeCombination("GatedMLP quantized weights are 2-D, 4-bit, group 64, bf16-scaled.");
            if (!aligned16(q->packedValues.data) || (reinterpret_cast<uintptr_t>(q->scales.data) & 3) ||
                (q->hasBiases && (reinterpret_cast<uintptr_t>(q->biases.data) & 3)))
                throw Error::invalidArgument("GatedMLP packed values must be 16-byte aligned, scales and biases 4-byte aligned");
        }
        F_ = wg.outFeatures();
        H_ = wg.inFeatures();
        if (wu.shape != wg.shape) throw Error::tensorShapeMismatch("GatedMLP up weight shape must match gate weight " + wg.shape.str() + ".");
        if (wd.shape != Shape({H_, F_}))
            throw Error::tensorShapeMismatch("GatedMLP down weight must be [" + std::to_string(H_) + ", " + std::to_string(F_) + "].");
        if (wg.hasBiases != wu.hasBiases) throw Error::invalidArgument("GatedMLP gate and up weights both have biases or neither");
        if (x.dataType != DataType::bf16 || out.dataType != DataType::bf16 || nw.dataType != DataType::f32)
            throw Error::unsupportedDataTypeCombination("GatedMLP with quantized weights takes bf16 x and out, an f32 norm weight.");
        if (H_ % 128 != 0 || F_ % 128 != 0 || H_ > 8192 || F_ > 16384)
            throw Error::tensorShapeMismatch("GatedMLP quantized: H, F multiples of 128, H <= 8192, F <= 16384.");
        if (x.shape.elementCount() != H_ || out.shape.elementCount() != H_)
            throw Error::tensorShapeMismatch("GatedMLP decodes one row: x and out hold [" + std::to_string(H_) + "].");
        requireElements(x, H_, "x");
        requireElements(nw, H_, "GatedMLP norm weight");
        for (const AffineQuantizedTensor *q : {&wg, &wu, &wd}) {
            const int64_t n = q->outFeatures(), k = q->inFeatures();
            requireElements(q->packedValues, n * (k / 8), "GatedMLP packed values");
            requireElements(q->scales, n * (k / 64), "GatedMLP scales");
            if (q->hasBiases) requireElements(q->biases, n * (k / 64), "GatedMLP biases");
        }
        if (hidden) {
            if (hidden->dataType != DataType::bf16) throw Error::unsupportedDataTypeCombination("GatedMLP hidden must be bf16.");
            requireElements(*hidden, F_, "GatedMLP hidden");
            h_ = *hidden;
            hasHidden_ = true;
        }
        lpr_ = q4Shape(F_, H_, false).lpr;
    }

    void setResidual(const Tensor &delta, const Tensor &wPost, const Tensor &xOut) {
        if (delta.dataType != DataType::bf16 || xOut.dataType != DataType::bf16 || wPost.dataType != DataType::f32)
            throw Error::unsupportedDataTypeCombination("GatedMLP residual: delta and x_out bf16, post-norm weight f32.");
        requireElements(delta, H_, "GatedMLP delta");
        requireElements(wPost, H_, "GatedMLP post-norm weight");
        requireElements(xOut, H_, "GatedMLP x_out");
        if (xOut.data == x_.data) throw Error::invalidArgument("GatedMLP x_out must not alias x (blocks read x while block 0 writes x_out)");
        delta_ = delta;
        wPost_ = wPost;
        xOut_ = xOut;
        residual_ = true;
    }

    std::vector<Binding> tensors() const override {
        std::vector<Binding> b = {{x_, kRead}, {nw_, kRead}, {out_, kWrite}};
        for (const AffineQuantizedTensor *q : {&wg_, &wu_, &wd_}) {
            b.push_back({q->packedValues, kRead});
            b.push_back({q->scales, kRead});
            if (q->hasBiases) b.push_back({q->biases, kRead});
        }
        if (hasHidden_) b.push_back({h_, kWrite});
        if (residual_) {
            b.push_back({delta_, kRead});
            b.push_back({wPost_, kRead});
            b.push_back({xOut_, kWrite});
        }
        return b;
    }

    std::string gateUpName() const {
        return "q4_gate_up_bf16_l" + std::to_string(lpr_) + (residual_ ? "_res" : "");
    }

    std::string describe() const override {
        // the down matvec reads the hidden tensor, or a 256-byte aligned scratch buffer
        void *hp = hasHidden_ ? h_.data : reinterpret_cast<void *>(uintptr_t{256});
        Tensor h(hp, Shape({1, F_}), DataType::bf16), o(out_.data, Shape({1, H_}), DataType::bf16);
        return gateUpName() + "," + Kernels::Matmul(h, wd_, o)->describe();
    }

    void encode(KernelCommandEncoder &enc) const override {
        auto run = [&](const Tensor &h) {
            GatedMLPConstants gc{(uint32_t)H_, (uint32_t)F_, 1u, 0u, eps_, (uint32_t)DataType::bf16, residual_ ? 1u : 0u};
            AffineQMatmulConstants qc{1u, (uint32_t)F_, (uint32_t)H_, (uint32_t)(H_ / 64), (uint32_t)(H_ / 8),
                                      wg_.hasBiases ? 1u : 0u};
            const Tensor d = residual_ ? delta_ : x_, w = residual_ ? wPost_ : x_, xo = residual_ ? xOut_ : x_;
            const size_t lds = (size_t)H_ * 4 + (size_t)(H_ / 64) * 36 * 4 + (size_t)(H_ / 64) * 4;
            FixedDispatch gu(gateUpName(),
                             {{x_, kRead}, {nw_, kRead}, {wg_.packedValues, kRead}, {wg_.scales, kRead},
                              {wg_.hasBiases ? wg_.biases : wg_.scales, kRead}, {wu_.packedValues, kRead}, {wu_.scales, kRead},
                              {wu_.hasBiases ? wu_.biases : wu_.scales, kRead}, {h, kWrite}, {d, kRead}, {w, kRead},
                              {xo, residual_ ? kWrite : kRead}},
                             {bytesOf(gc), bytesOf(qc)}, grid1(streamBlocks(cdiv(F_, 64 / lpr_)), kBlock, lds));
            enc.dispatch(gu);
            Tensor hv(h.data, Shape({1, F_}), DataType::bf16), ov(out_.data, Shape({1, H_}), DataType::bf16);
            Kernels::Matmul(hv, wd_, ov)->encode(enc);
        };
        if (hasHidden_) {
            run(h_);
        } else {
            enc.withTemporaryTensor(ScratchSpec{{F_}, DataType::bf16}, [&](Tensor h) { run(h); });
        }
    }

private:
    Tensor x_, nw_;
    AffineQuantizedTensor wg_, wu_, wd_;
    Tensor out_, h_, delta_, wPost_, xOut_;
    float eps_;
    bool hasHidden_ = false, residual_ = false;
    int64_t H_ = 0, F_ = 0;
    int lpr_ = 8;
};

// ---------------------------------------------------------------------------
// Argmax (Argmax.swift) as two stages over row slices
// ---------------------------------------------------------------------------

class ArgmaxKernel : public Kernel {
public:
    ArgmaxKernel(const Tensor &x, const Tensor &indices, int64_t rows, int64_t n) : x_(x), idx_(indices), rows_(rows), n_(n) {
        if (x.dataType != DataType::f32) throw Error::unsupportedDataTypeCombination("Argmax reads f32 values.");
        if (indices.dataType != DataType::i32) throw Error::unsupportedDataTypeCombination("Argmax indices are i32.");
        if (n <= 0) throw Error::tensorShapeMismatch("Argmax needs a non-empty axis.");
        requireElements(x, rows * n, "Argmax x");
        requireElements(indices, rows, "Argmax indices");
        slices_ = std::clamp<int64_t>(cdiv(n, 4096), 1, 256);
    }
    std::vector<Binding> tensors() const override { return {{x_, kRead}, {idx_, kWrite}}; }
    std::string describe() const override { return "argmax_partial,argmax_finish"; }
    void encode(KernelCommandEncoder &enc) const override {
        if (rows_ == 0) return;
        ArgmaxSliceConstants ac{(uint32_t)rows_, (uint32_t)n_, (uint32_t)slices_};
        enc.withTemporaryTensor(ScratchSpec{{rows_ * slices_}, DataType::f32}, [&](Tensor pv) {
            enc.withTemporaryTensor(ScratchSpec{{rows_ * slices_}, DataType::i32}, [&](Tensor pi) {
                DispatchSize ds;
                ds.grid = dim3((unsigned)slices_, (unsigned)rows_, 1);
                ds.block = dim3(kBlock, 1, 1);
                FixedDispatch s1("argmax_partial", {{x_, kRead}, {pv, kWrite}, {pi, kWrite}}, {bytesOf(ac)}, ds);
                enc.dispatch(s1);
                FixedDispatch s2("argmax_finish", {{x_, kRead}, {pv, kRead}, {pi, kRead}, {idx_, kWrite}}, {bytesOf(ac)},
                                 grid1(rows_, kBlock));
                enc.dispatch(s2);
            });
        });
    }

private:
    Tensor x_, idx_;
    int64_t rows_, n_, slices_ = 1;
};

std::unique_ptr<Kernel> elementwise(const char *base, const Tensor &a, const Tensor *b, const Tensor &out,
                                    std::vector<uint8_t> consts) {
    if (!isFloat(a.dataType)) throw Error::unsupportedDataTypeCombination(std::string("Unsupported ") + base + " data type: " + tag(a.dataType) + ".");
    if (out.dataType != a.dataType || (b && b->dataType != a.dataType))
        throw Error::unsupportedDataTypeCombination(std::string(base) + " needs one dtype for inputs and output.");
    const int64_t count = a.shape.elementCount();
    requireElements(a, count, base);
    requireElements(out, count, base);
    if (b) requireElements(*b, count, base);
    std::string fn = base;
    if (a.dataType != DataType::f32) fn += std::string("_") + tag(a.dataType);
    std::vector<Binding> binds = {{a, kRead}};
    if (b) binds.push_back({*b, kRead});
    binds.push_back({out, kWrite});
    const int64_t blocks = std::clamp<int64_t>(cdiv(cdiv(count, 16 / stride(a.dataType)), kBlock), 1, 8 * deviceCUs());
    return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{std::move(consts)}, grid1(blocks, kBlock));
}

}  // namespace

// AffineQuantizedTensor.swift:29-48, plus the format's own consistency (bits
// dividing the 32-bit word, a positive group size).
void AffineQuantizedTensor::validate() const {
    if (shape.rank() < 2) throw Error::tensorInvalidRank(2, shape.rank());
    if (hasBiases) {
        if (biases.dataType != scales.dataType)
            throw Error::unsupportedDataTypeCombination(std::string("AffineQuantizedTensor scales and biases must share a data type; got ") +
                                                        name(scales.dataType) + " and " + name(biases.dataType) + ".");
        if (biases.shape != scales.shape)
            throw Error::tensorShapeMismatch("AffineQuantizedTensor scales and biases must share a shape; got " + scales.shape.str() +
                                             " and " + biases.shape.str() + ".");
    }
    if (packedValues.dataType != DataType::u32)
        throw Error::unsupportedDataTypeCombination(
            std::string("AffineQuantizedTensor packed values must use u32 for packing uint32LittleEndian; got ") +
            name(packedValues.dataType) + ".");
    if (bits <= 0 || bits > 32 || 32 % bits != 0 || groupSize <= 0)
        throw Error::invalidArgument("AffineQuantizedTensor format needs bits dividing 32 and a positive group size.");
}

namespace Kernels {

// FlashAttention.swift:109-113: one query row -> split-KV decoding; 32 rows
// or more with a head dim up to 512 -> the tiled kernel on the matrix cores
// (where the reference takes MPP); otherwise the plain per-row kernel.
AttentionPath route(int64_t queryLen, int64_t headDim, DataType qType) {
    if (queryLen == 1) return AttentionPath::decoding;
    const bool sixteen = qType == DataType::f16 || qType == DataType::bf16;
    // the matrix-core kernels take any head dim up to 512 in 16-byte rows,
    // padded to 64, 128, 256 or 512 inside (MPPFlashAttention's hd256 and
    // hd512 buckets, FlashAttention.swift:305-311), in f16, bf16 and f32
    const int64_t perChunk = sixteen ? 8 : 4;
    if (queryLen >= 32 && (sixteen || qType == DataType::f32) && headDim <= 512 && headDim % perChunk == 0)
        return AttentionPath::tiled;
    return AttentionPath::plain;
}

// FlashAttention.swift:51-90
std::unique_ptr<Kernel> FlashAttention(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, float scale,
                                       AttentionMask mask) {
    if (q.shape.rank() != 4) throw Error::tensorInvalidRank(4, q.shape.rank());
    if (k.shape.rank() != 4) throw Error::tensorInvalidRank(4, k.shape.rank());
    if (v.shape.rank() != 4) throw Error::tensorInvalidRank(4, v.shape.rank());
    const int64_t B = q.shape[0], Nq = q.shape[1], Sq = q.shape[2], Hd = q.shape[3];
    const int64_t Nkv = k.shape[1], Sk = k.shape[2];
    if (k.shape[0] != B || k.shape[3] != Hd)
        throw Error::tensorShapeMismatch("FlashAttention K shape must match Q batch/headDim; q " + q.shape.str() + ", k " + k.shape.str() + ".");
    if (v.shape != k.shape)
        throw Error::tensorShapeMismatch("FlashAttention V shape must match K; v " + v.shape.str() + ", k " + k.shape.str() + ".");
    if (out.shape != Shape({B, Nq, Sq, Hd}))
        throw Error::tensorShapeMismatch("FlashAttention output shape must be " + Shape({B, Nq, Sq, Hd}).str() + "; got " + out.shape.str() + ".");
    return std::make_unique<FlashAttentionKernel>(q, k, v, out, AttnDims{B, Nq, Nkv, Sq, Sk, Hd, Sk}, scale, mask, nullptr);
}

// FlashAttention.swift:13-49, plus key capacity and position
std::unique_ptr<Kernel> FlashAttention(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, int64_t batch,
                                       int64_t queryHeads, int64_t kvHeads, int64_t queryLen, int64_t keyLen, int64_t headDim,
                                       float scale, AttentionMask mask, int64_t keyCapacity, const Tensor *position) {
    const int64_t cap = keyCapacity > 0 ? keyCapacity : keyLen;
    return std::make_unique<FlashAttentionKernel>(q, k, v, out, AttnDims{batch, queryHeads, kvHeads, queryLen, keyLen, headDim, cap},
                                                  scale, mask, position);
}

// The split-KV attention with its partials in the static scratch
// (static_scratch.hip) instead of a borrowed buffer: validation and kernels
// as for FlashAttention with the same dims; no device memory is allocated.
void FlashDecodingNoAlloc(KernelLibrary &library, hipStream_t stream, const Tensor &q, const Tensor &k, const Tensor &v,
                          const Tensor &out, int64_t batch, int64_t queryHeads, int64_t kvHeads, int64_t queryLen,
                          int64_t keyLen, int64_t headDim, float scale, AttentionMask mask, int64_t keyCapacity,
                          const Tensor *position) {
    struct NoScratch : KernelScratchAllocator {
        KernelTemporaryBuffer borrowTemporaryBuffer(size_t) override {
            throw Error(POPCORN_ERR_WORKSPACE_EXHAUSTED, "the allocation-free attention borrows no scratch");
        }
    } none;
    const int64_t cap = keyCapacity > 0 ? keyCapacity : keyLen;
    FlashAttentionKernel fa(q, k, v, out, AttnDims{batch, queryHeads, kvHeads, queryLen, keyLen, headDim, cap}, scale,
                            mask, position);
    fa.useSplitPath();
    size_t bytes = 0;
    void *scratch = staticScratch(&bytes);
    KernelCommandEncoder enc(library, stream, none);
    fa.encodeSplitInto(enc, scratch, bytes);
}

// Matmul.swift:68-93
std::unique_ptr<Kernel> Matmul(const Tensor &a, const Tensor &b, const Tensor &c, bool transposeB) {
    if (a.shape.rank() != 2) throw Error::tensorInvalidRank(2, a.shape.rank());
    if (b.shape.rank() != 2) throw Error::tensorInvalidRank(2, b.shape.rank());
    if (c.shape.rank() != 2) throw Error::tensorInvalidRank(2, c.shape.rank());
    const int64_t m = a.shape[0], k = a.shape[1];
    const int64_t n = transposeB ? b.shape[0] : b.shape[1];
    const Shape expectedB = transposeB ? Shape({n, k}) : Shape({k, n});
    if (b.shape != expectedB)
        throw Error::tensorShapeMismatch("Matmul RHS shape mismatch: expected " + expectedB.str() + ", got " + b.shape.str() + ".");
    if (c.shape != Shape({m, n}))
        throw Error::tensorShapeMismatch("Matmul output shape mismatch: expected " + Shape({m, n}).str() + ", got " + c.shape.str() + ".");
    return makeMatmul(a, b, c, m, k, n, transposeB);
}

std::unique_ptr<Kernel> Matmul(const Tensor &a, const Tensor &b, const Tensor &c, int64_t m, int64_t k, int64_t n, bool transposeB) {
    return makeMatmul(a, b, c, m, k, n, transposeB);
}

// RMSNorm.swift:10-37
std::unique_ptr<Kernel> RMSNorm(const Tensor &x, const Tensor *weight, const Tensor &out, int64_t rowCount, int64_t hiddenSize,
                                float eps, bool addOneToWeight) {
    const char *fn = nullptr;
    switch (x.dataType) {
    case DataType::f32: fn = "rmsnorm"; break;
    case DataType::f16: fn = "rmsnorm_f16"; break;
    case DataType::bf16: fn = "rmsnorm_bf16"; break;
    default: throw Error::unsupportedDataTypeCombination(std::string("Unsupported RMSNorm data type: ") + tag(x.dataType) + ".");
    }
    if (out.dataType != x.dataType) throw Error::unsupportedDataTypeCombination("RMSNorm output must have the input's dtype.");
    if (weight && weight->dataType != DataType::f32)
        throw Error::unsupportedDataTypeCombination("RMSNorm weight must be f32 (RMSNorm.metal:42-46 reads it as float).");
    if (hiddenSize <= 0 || rowCount < 0) throw Error::tensorShapeMismatch("RMSNorm needs a positive hidden size.");
    requireElements(x, rowCount * hiddenSize, "RMSNorm x");
    requireElements(out, rowCount * hiddenSize, "RMSNorm out");
    if (weight) requireElements(*weight, hiddenSize, "RMSNorm weight");
    RMSNormConstants rc{(uint32_t)hiddenSize, weight ? 1u : 0u, addOneToWeight ? 1u : 0u, eps};
    // From 8 rows on, rows of whole 16-byte vectors, up to 1024 of them: 16, 32
    // or 64 lanes per row (rmsnorm_lanes; 8 rows of 2304, bf16: 3.5 us against
    // 3.9 on a block per row; fewer rows keep that). Blocks of one wave for
    // 64-lane rows and where four would leave CUs idle (1000 x 2304: 4.4
    // against 4.6 us; 8000 x 256: 3.5 against 3.25). Long f32 rows, whose block
    // loads a vector per lane, keep a block per row while there are no more of
    // them than the CUs hold (f32, us block per row and lanes: 8 x 1536 equal, 8
    // x 2304 3.2 and 4.0, 200 x 2304 3.5 and 4.2, 256 x 2304 4.8 and 4.3; 200 x
    // 4096 4.4 and 5.6, 300 x 4096 6.1 and 6.3, 600 x 4096 7.9 and 7.2).
    const int64_t perVec = 16 / stride(x.dataType), nvec = cdiv(hiddenSize, perVec);
    const bool longF32 = x.dataType == DataType::f32 && nvec >= 384 && rowCount < (nvec > 768 ? 2 : 1) * (int64_t)deviceCUs();
    if (rowCount >= 8 && hiddenSize % perVec == 0 && nvec <= 1024 && !longF32 && aligned16(x.data) && aligned16(out.data) &&
        (!weight || aligned16(weight->data)) && rowCount <= UINT32_MAX) {
        const int64_t lanes = nvec <= 16 ? 16 : nvec <= 32 ? 32 : 64;
        const int vectors = nvec <= 64 ? 1 : nvec <= 256 ? 4 : nvec <= 512 ? 8 : 16;
        const int threads = lanes == 64 || rowCount * lanes < kBlock * (int64_t)deviceCUs() ? 64 : kBlock;
        const uint32_t rows = (uint32_t)rowCount;
        return std::make_unique<FixedDispatch>(
            std::string("rmsnorm_rows_") + tag(x.dataType) + "_l" + std::to_string(lanes) + "_v" + std::to_string(vectors),
            std::vector<Binding>{{x, kRead}, {weight ? *weight : x, kRead}, {out, kWrite}},
            std::vector<std::vector<uint8_t>>{bytesOf(rc), bytesOf(rows)}, grid1(cdiv(rowCount, threads / lanes), threads));
    }
    // One block per row; a lone row spreads over more lanes (latency), many
    // rows use 256 threads.
    int threads = kBlock;
    if (rowCount < deviceCUs()) threads = (int)std::clamp<int64_t>(cdiv(nvec, 64) * 64, 64, 1024);
    const Tensor &w = weight ? *weight : x;  // RMSNorm.swift:21: x bound as the absent weight
    return std::make_unique<FixedDispatch>(fn, std::vector<Binding>{{x, kRead}, {w, kRead}, {out, kWrite}},
                                           std::vector<std::vector<uint8_t>>{bytesOf(rc)}, grid1(rowCount, threads));
}

// RMSNorm.swift:39-70
std::unique_ptr<Kernel> RMSNorm(const Tensor &x, const Tensor *weight, const Tensor &out, int axis, float eps, bool addOneToWeight) {
    const int rank = x.shape.rank();
    const int norm = axis < 0 ? rank + axis : axis;
    if (norm != rank - 1 || rank <= 0) throw Error::tensorInvalidAxis(axis, rank);
    if (x.shape != out.shape)
        throw Error::tensorShapeMismatch("RMSNorm output shape must match input; got " + out.shape.str() + ", expected " + x.shape.str() + ".");
    const int64_t H = x.shape[norm];
    const int64_t rows = H ? x.shape.elementCount() / H : 0;
    if (weight && !(weight->shape == Shape({H}) || weight->shape == x.shape))
        throw Error::tensorShapeMismatch("RMSNorm weight shape must be [" + std::to_string(H) + "] or " + x.shape.str() + "; got " +
                                         weight->shape.str() + ".");
    return RMSNorm(x, weight, out, rows, H, eps, addOneToWeight);
}

// KVCacheWrite.swift:7-35, plus f16 and a run-time position
std::unique_ptr<Kernel> KVCacheWrite(const Tensor &source, const Tensor &cache, int64_t batch, int64_t kvHeads, int64_t newLen,
                                     int64_t maxLen, int64_t headDim, int64_t offset, const Tensor *position) {
    using D = DataType;
    const D s = source.dataType, c = cache.dataType;
    const char *fn = nullptr;
    if (s == D::f32 && c == D::f32) fn = "kv_cache_write";
    else if (s == D::bf16 && c == D::bf16) fn = "kv_cache_write_bf16";
    else if (s == D::f32 && c == D::bf16) fn = "kv_cache_write_f32_to_bf16";
    else if (s == D::f16 && c == D::f16) fn = "kv_cache_write_f16";
    else
        throw Error::unsupportedDataTypeCombination(std::string("Unsupported KV cache data type combination: ") + tag(s) + ", " + tag(c) + ".");
    if (batch < 0 || kvHeads < 0 || newLen < 0 || headDim <= 0 || maxLen < 0)
        throw Error::tensorShapeMismatch("KV cache write dimensions must be non-negative.");
    if (!position && (offset < 0 || offset + newLen > maxLen))
        throw Error::tensorShapeMismatch("KV cache write range " + std::to_string(offset) + "..<" + std::to_string(offset + newLen) +
                                         " exceeds cache length " + std::to_string(maxLen) + ".");
    requireElements(source, batch * kvHeads * newLen * headDim, "KV cache source");
    requireElements(cache, batch * kvHeads * maxLen * headDim, "KV cache");
    if (position) {
        if (position->dataType != D::i32) throw Error::unsupportedDataTypeCombination("position tensor must be i32");
        requireElements(*position, 1, "position");
    }
    const int64_t run = 16 / stride(s);
    const int64_t runs = batch * kvHeads * newLen * cdiv(headDim, run);
    const int64_t blocks = std::clamp<int64_t>(cdiv(runs, kBlock), 1, 4096);
    if (!position) {
        // the reference's kernel and constants (KVCacheWrite.metal:6-11)
        KVCacheWriteConstants kc{(uint32_t)batch, (uint32_t)kvHeads, (uint32_t)newLen, (uint32_t)maxLen,
                                 (uint32_t)headDim, (uint32_t)offset};
        return std::make_unique<FixedDispatch>(fn, std::vector<Binding>{{source, kRead}, {cache, kWrite}},
                                               std::vector<std::vector<uint8_t>>{bytesOf(kc)},
                                               grid1(runs ? blocks : 0, kBlock));
    }
    KVCacheWriteExtConstants kc{(uint32_t)batch, (uint32_t)kvHeads, (uint32_t)newLen, (uint32_t)maxLen, (uint32_t)headDim,
                                (uint32_t)std::max<int64_t>(offset, 0), 1u};
    return std::make_unique<FixedDispatch>(std::string(fn) + "_ext",
                                           std::vector<Binding>{{source, kRead}, {cache, kWrite}, {*position, kRead}},
                                           std::vector<std::vector<uint8_t>>{bytesOf(kc)}, grid1(runs ? blocks : 0, kBlock));
}

// KVCacheWrite.swift:37-48
std::unique_ptr<Kernel> KVCacheWrite(const Tensor &source, const Tensor &cache, int64_t offset) {
    if (source.shape.rank() != 4) throw Error::tensorInvalidRank(4, source.shape.rank());
    if (cache.shape.rank() != 4) throw Error::tensorInvalidRank(4, cache.shape.rank());
    const int64_t B = source.shape[0], Nkv = source.shape[1], Snew = source.shape[2], Hd = source.shape[3];
    if (cache.shape[0] != B || cache.shape[1] != Nkv || cache.shape[3] != Hd)
        throw Error::tensorShapeMismatch("KV cache shape must match source batch/heads/headDim; source " + source.shape.str() +
                                         ", cache " + cache.shape.str() + ".");
    if (offset < 0 || offset + Snew > cache.shape[2])
        throw Error::tensorShapeMismatch("KV cache write range " + std::to_string(offset) + "..<" + std::to_string(offset + Snew) +
                                         " exceeds cache length " + std::to_string(cache.shape[2]) + ".");
    return KVCacheWrite(source, cache, B, Nkv, Snew, cache.shape[2], Hd, offset, nullptr);
}

// GeluTanh.swift:28-33
std::unique_ptr<Kernel> GeluTanh(const Tensor &x, const Tensor &out) {
    if (x.shape != out.shape)
        throw Error::tensorShapeMismatch("GeluTanh output shape must match input; got " + out.shape.str() + ", expected " + x.shape.str() + ".");
    return elementwise("gelu_tanh", x, nullptr, out, bytesOf(GeluTanhConstants{(uint32_t)x.shape.elementCount()}));
}

// Mul.swift:28-37
std::unique_ptr<Kernel> Mul(const Tensor &a, const Tensor &b, const Tensor &out) {
    if (a.shape != b.shape) throw Error::tensorShapeMismatch("Mul requires matching input shapes; got " + a.shape.str() + " and " + b.shape.str() + ".");
    if (a.shape != out.shape) throw Error::tensorShapeMismatch("Mul output shape must match inputs; got " + out.shape.str() + ", expected " + a.shape.str() + ".");
    return elementwise("mul", a, &b, out, bytesOf(MulConstants{(uint32_t)a.shape.elementCount()}));
}

// Add.swift
std::unique_ptr<Kernel> Add(const Tensor &a, const Tensor &b, const Tensor &out) {
    if (a.shape != b.shape) throw Error::tensorShapeMismatch("Add requires matching input shapes; got " + a.shape.str() + " and " + b.shape.str() + ".");
    if (a.shape != out.shape) throw Error::tensorShapeMismatch("Add output shape must match inputs; got " + out.shape.str() + ", expected " + a.shape.str() + ".");
    return elementwise("add", a, &b, out, bytesOf(AddConstants{(uint32_t)a.shape.elementCount()}));
}

// ScalarMul.swift
std::unique_ptr<Kernel> ScalarMul(const Tensor &x, float scalar, const Tensor &out) {
    if (x.shape != out.shape)
        throw Error::tensorShapeMismatch("ScalarMul output shape must match input; got " + out.shape.str() + ", expected " + x.shape.str() + ".");
    return elementwise("scalar_mul", x, nullptr, out, bytesOf(ScalarMulConstants{(uint32_t)x.shape.elementCount(), scalar}));
}

// RopeBuildCosSin.swift:8-28: positions i32 [T], inv_freq f32 [Hd2] -> cos,
// sin f32 [T, Hd2] (the Metal kernel's buffer types, checked here).
std::unique_ptr<Kernel> RopeBuildCosSin(const Tensor &positions, const Tensor &invFreq, const Tensor &cosOut,
                                        const Tensor &sinOut, int64_t seqLen, int64_t halfHeadDim, float scaling) {
    if (positions.dataType != DataType::i32) throw Error::unsupportedDataTypeCombination("RoPE positions must be i32.");
    if (invFreq.dataType != DataType::f32 || cosOut.dataType != DataType::f32 || sinOut.dataType != DataType::f32)
        throw Error::unsupportedDataTypeCombination("RoPE invFreq and the cos/sin tables are f32.");
    if (seqLen < 0 || halfHeadDim < 0 || seqLen > UINT32_MAX || halfHeadDim > UINT32_MAX)
        throw Error::tensorShapeMismatch("RoPE table dimensions out of range.");
    requireElements(positions, seqLen, "RoPE positions");
    requireElements(invFreq, halfHeadDim, "RoPE invFreq");
    requireElements(cosOut, seqLen * halfHeadDim, "RoPE cos");
    requireElements(sinOut, seqLen * halfHeadDim, "RoPE sin");
    RopeBuildCosSinConstants c{(uint32_t)seqLen, (uint32_t)halfHeadDim, scaling};
    const int64_t n = seqLen * halfHeadDim;
    const int64_t blocks = n ? std::clamp<int64_t>(cdiv(n, kBlock), 1, 8 * deviceCUs()) : 0;
    return std::make_unique<FixedDispatch>(
        "rope_build_cos_sin",
        std::vector<Binding>{{positions, kRead}, {invFreq, kRead}, {cosOut, kWrite}, {sinOut, kWrite}},
        std::vector<std::vector<uint8_t>>{bytesOf(c)}, grid1(blocks, kBlock));
}

// RopeBuildCosSin.swift:30-50
std::unique_ptr<Kernel> RopeBuildCosSin(const Tensor &positions, const Tensor &invFreq, const Tensor &cosOut,
                                        const Tensor &sinOut, float scaling) {
    if (cosOut.shape != sinOut.shape)
        throw Error::tensorShapeMismatch("RoPE cos and sin output shapes must match; got " + cosOut.shape.str() + " and " +
                                         sinOut.shape.str() + ".");
    if (cosOut.shape.rank() != 2) throw Error::tensorInvalidRank(2, cosOut.shape.rank());
    const int64_t seqLen = cosOut.shape[0], halfHeadDim = cosOut.shape[1];
    if (positions.shape.elementCount() != seqLen)
        throw Error::tensorShapeMismatch("RoPE positions count must equal seqLen " + std::to_string(seqLen) + "; got " +
                                         std::to_string(positions.shape.elementCount()) + ".");
    if (invFreq.shape.elementCount() != halfHeadDim)
        throw Error::tensorShapeMismatch("RoPE invFreq count must equal halfHeadDim " + std::to_string(halfHeadDim) +
                                         "; got " + std::to_string(invFreq.shape.elementCount()) + ".");
    return RopeBuildCosSin(positions, invFreq, cosOut, sinOut, seqLen, halfHeadDim, scaling);
}

// RopeApply.swift:8-44: x [B, T, Nh, Hd] with tables [T, Hd/2]; the function
// is chosen by (x, table) dtypes as the reference does (:25-30); out has x's
// dtype.
std::unique_ptr<Kernel> RopeApply(const Tensor &x, const Tensor &cosT, const Tensor &sinT, const Tensor &out,
                                  int64_t batch, int64_t seqLen, int64_t headCount, int64_t headDim) {
    if (headDim % 2 != 0)
        throw Error::tensorShapeMismatch("RoPE head dimension must be even; got " + std::to_string(headDim) + ".");
    const char *fn = nullptr;
    if (x.dataType == DataType::f32 && cosT.dataType == DataType::f32) fn = "rope_apply";
    else if (x.dataType == DataType::bf16 && cosT.dataType == DataType::bf16) fn = "rope_apply_bf16";
    else if (x.dataType == DataType::bf16 && cosT.dataType == DataType::f32) fn = "rope_apply_f32_tables_bf16";
    else
        throw Error::unsupportedDataTypeCombination(std::string("Unsupported RoPE data type combination: ") + tag(x.dataType) +
                                                    ", " + tag(cosT.dataType) + ".");
    if (sinT.dataType != cosT.dataType || out.dataType != x.dataType)
        throw Error::unsupportedDataTypeCombination("RoPE sin table must match cos, and out must match x.");
    if (batch < 0 || seqLen < 0 || headCount < 0 || headDim < 0 || batch > UINT32_MAX || seqLen > UINT32_MAX ||
        headCount > UINT32_MAX || headDim > UINT32_MAX)
        throw Error::tensorShapeMismatch("RoPE dimensions out of range.");
    const int64_t n = batch * seqLen * headCount * headDim;
    requireElements(x, n, "RoPE x");
    requireElements(out, n, "RoPE out");
    requireElements(cosT, seqLen * (headDim / 2), "RoPE cos");
    requireElements(sinT, seqLen * (headDim / 2), "RoPE sin");
    RopeApplyConstants c{(uint32_t)batch, (uint32_t)seqLen, (uint32_t)headCount, (uint32_t)(headDim / 2)};
    const int64_t items = batch * seqLen * headCount * cdiv(headDim / 2, 8);
    const int64_t blocks = items ? std::clamp<int64_t>(cdiv(items, kBlock), 1, 8 * deviceCUs()) : 0;
    return std::make_unique<FixedDispatch>(
        fn, std::vector<Binding>{{x, kRead}, {cosT, kRead}, {sinT, kRead}, {out, kWrite}},
        std::vector<std::vector<uint8_t>>{bytesOf(c)}, grid1(blocks, kBlock));
}

// RopeApply.swift:46-60
std::unique_ptr<Kernel> RopeApply(const Tensor &x, const Tensor &cosT, const Tensor &sinT, const Tensor &out) {
    if (x.shape.rank() != 4) throw Error::tensorInvalidRank(4, x.shape.rank());
    if (x.shape != out.shape)
        throw Error::tensorShapeMismatch("RoPE output shape must match input; got " + out.shape.str() + ", expected " +
                                         x.shape.str() + ".");
    const int64_t batch = x.shape[0], seqLen = x.shape[1], headCount = x.shape[2], headDim = x.shape[3];
    if (headDim % 2 != 0)
        throw Error::tensorShapeMismatch("RoPE head dimension must be even; got " + std::to_string(headDim) + ".");
    const Shape table{seqLen, headDim / 2};
    if (cosT.shape != table || sinT.shape != table)
        throw Error::tensorShapeMismatch("RoPE tables must have shape " + table.str() + "; got cos " + cosT.shape.str() +
                                         ", sin " + sinT.shape.str() + ".");
    return RopeApply(x, cosT, sinT, out, batch, seqLen, headCount, headDim);
}

// Transpose12.swift:8-25: [D0, D1, D2, D3] -> [D0, D2, D1, D3].
std::unique_ptr<Kernel> Transpose12(const Tensor &src, const Tensor &out, int64_t d0, int64_t d1, int64_t d2, int64_t d3) {
    const char *fn = nullptr;
    switch (src.dataType) {
    case DataType::f32: fn = "transpose12"; break;
    case DataType::f16: fn = "transpose12_f16"; break;
    case DataType::bf16: fn = "transpose12_bf16"; break;
    default:
        throw Error::unsupportedDataTypeCombination(std::string("Unsupported transpose12 data type: ") + tag(src.dataType) + ".");
    }
    if (out.dataType != src.dataType) throw Error::unsupportedDataTypeCombination("Transpose12 output must match the source dtype.");
    for (int64_t d : {d0, d1, d2, d3})
        if (d < 0 || d > UINT32_MAX) throw Error::tensorShapeMismatch("Transpose12 dimensions out of range.");
    const int64_t n = d0 * d1 * d2 * d3;
    requireElements(src, n, "Transpose12 src");
    requireElements(out, n, "Transpose12 out");
    Transpose12Constants c{(uint32_t)d0, (uint32_t)d1, (uint32_t)d2, (uint32_t)d3};
    const int64_t runs = (d3 % (16 / stride(src.dataType)) == 0) ? n / (16 / stride(src.dataType)) : n;
    const int64_t blocks = runs ? std::clamp<int64_t>(cdiv(runs, kBlock), 1, 8 * deviceCUs()) : 0;
    return std::make_unique<FixedDispatch>(fn, std::vector<Binding>{{src, kRead}, {out, kWrite}},
                                           std::vector<std::vector<uint8_t>>{bytesOf(c)}, grid1(blocks, kBlock));
}

// Transpose12.swift:27-35
std::unique_ptr<Kernel> Transpose12(const Tensor &src, const Tensor &out) {
    if (src.shape.rank() != 4) throw Error::tensorInvalidRank(4, src.shape.rank());
    const int64_t d0 = src.shape[0], d1 = src.shape[1], d2 = src.shape[2], d3 = src.shape[3];
    const Shape expected{d0, d2, d1, d3};
    if (out.shape != expected)
        throw Error::tensorShapeMismatch("Transpose12 output shape must be " + expected.str() + "; got " + out.shape.str() + ".");
    return Transpose12(src, out, d0, d1, d2, d3);
}

std::unique_ptr<Kernel> GatedMLP(const Tensor &x, const Tensor *normWeight, const Tensor &wGate, const Tensor &wUp,
                                 const Tensor &wDown, const Tensor &out, float eps, bool addOneToWeight, const Tensor *hidden) {
    return std::make_unique<GatedMLPKernel>(x, normWeight, wGate, wUp, wDown, out, eps, addOneToWeight, hidden);
}

std::unique_ptr<Kernel> GatedMLPResidual(const Tensor &xIn, const Tensor &delta, const Tensor &wPost, const Tensor &xOut,
                                         const Tensor *normWeight, const Tensor &wGate, const Tensor &wUp,
                                         const Tensor &wDown, const Tensor &out, float eps, bool addOneToWeight,
                                         const Tensor *hidden) {
    auto k = std::make_unique<GatedMLPKernel>(xIn, normWeight, wGate, wUp, wDown, out, eps, addOneToWeight, hidden);
    k->setResidual(delta, wPost, xOut);
    return k;
}

std::unique_ptr<Kernel> DecodeAttention(const DecodeAttentionArgs &a) { return std::make_unique<DecodeAttentionKernel>(a); }

std::unique_ptr<Kernel> GatedMLPResidual(const Tensor &xIn, const Tensor *delta, const Tensor *wPost, const Tensor *xOut,
                                         const Tensor &normWeight, const AffineQuantizedTensor &wGate,
                                         const AffineQuantizedTensor &wUp, const AffineQuantizedTensor &wDown, const Tensor &out,
                                         float eps, const Tensor *hidden) {
    auto k = std::make_unique<GatedMLPQ4Kernel>(xIn, normWeight, wGate, wUp, wDown, out, eps, hidden);
    if (delta || wPost || xOut) {
        if (!delta || !wPost || !xOut) throw Error::invalidArgument("the residual form needs delta, w_post and x_out");
        k->setResidual(*delta, *wPost, *xOut);
    }
    return k;
}

std::unique_ptr<Kernel> DecodeMatvec(const DecodeMatvecArgs &a) {
    if (!a.x || !(a.weight || a.qweight) || !a.out) throw Error::invalidArgument("DecodeMatvec needs x, a weight and out");
    if (a.weight && a.qweight) throw Error::invalidArgument("DecodeMatvec takes a dense or a quantized weight, not both");
    const bool q4 = a.qweight != nullptr;
    int64_t N = 0, K = 0;
    DataType t;
    if (q4) {
        const AffineQuantizedTensor &Q = *a.qweight;
        Q.validate();
        N = Q.outFeatures();
        K = Q.inFeatures();
        t = a.x->dataType;
        if (t != DataType::bf16 || Q.bits != 4 || Q.groupSize != 64 || Q.scales.dataType != DataType::bf16)
            throw Error::unsupportedDataTypeCombination("DecodeMatvec with a quantized weight takes bf16 x and a 4-bit, group-64, "
                                                        "bf16-scaled weight.");
        if (K <= 0 || N <= 0 || K % 128 != 0 || K > 8192)
            throw Error::tensorShapeMismatch("DecodeMatvec with a quantized weight needs K a multiple of 128, 0 < K <= 8192.");
        requireElements(Q.packedValues, N * (K / 8), "DecodeMatvec packed values");
        requireElements(Q.scales, N * (K / 64), "DecodeMatvec scales");
        if (Q.hasBiases) requireElements(Q.biases, N * (K / 64), "DecodeMatvec biases");
        if (!aligned16(Q.packedValues.data) || (reinterpret_cast<uintptr_t>(Q.scales.data) & 3) ||
            (Q.hasBiases && (reinterpret_cast<uintptr_t>(Q.biases.data) & 3)))
            throw Error::invalidArgument("DecodeMatvec packed values must be 16-byte aligned, scales and biases 4-byte aligned");
    } else {
        const Tensor &W = *a.weight;
        if (W.shape.rank() != 2) throw Error::tensorInvalidRank(2, W.shape.rank());
        N = W.shape[0];
        K = W.shape[1];
        t = W.dataType;
        if (!isFloat(t) || a.x->dataType != t)
            throw Error::unsupportedDataTypeCombination("DecodeMatvec needs x and weight of one float dtype.");
        if (K <= 0 || N <= 0 || K > kMaxStagedK) throw Error::tensorShapeMismatch("DecodeMatvec needs 0 < K <= 16384 and N > 0.");
        requireElements(W, N * K, "DecodeMatvec weight");
    }
    const DataType o = a.out->dataType;
    if (!(o == t || o == DataType::f32)) throw Error::unsupportedDataTypeCombination("DecodeMatvec output is the weight dtype or f32.");
    requireElements(*a.x, K, "DecodeMatvec x");
    uint32_t flags = 0;
    if (a.delta) {
        if (!a.wPost || !a.xOut) throw Error::invalidArgument("DecodeMatvec with delta needs wPost and xOut");
        if (a.delta->dataType != t || a.xOut->dataType != t || a.wPost->dataType != DataType::f32)
            throw Error::unsupportedDataTypeCombination("DecodeMatvec residual: delta and xOut of x's dtype, wPost f32.");
        requireElements(*a.delta, K, "DecodeMatvec delta");
        requireElements(*a.wPost, K, "DecodeMatvec wPost");
        requireElements(*a.xOut, K, "DecodeMatvec xOut");
        if (a.xOut->data == a.x->data) throw Error::invalidArgument("DecodeMatvec xOut must not alias x");
        flags |= 1u;
    }
    if (a.wPre) {
        if (a.wPre->dataType != DataType::f32) throw Error::unsupportedDataTypeCombination("DecodeMatvec wPre must be f32.");
        requireElements(*a.wPre, K, "DecodeMatvec wPre");
        flags |= 2u;
    }
    DecodeMatvecConstants dc{(uint32_t)K, (uint32_t)N, a.eps, 0u, (uint32_t)t, (uint32_t)N, 0u, 1u, 1u};
    if (a.kCache || a.vCache) {
        if (!a.kCache || !a.vCache || !a.position) throw Error::invalidArgument("KV scatter needs both caches and a position");
        const Tensor &kc = *a.kCache;
        if (kc.shape != a.vCache->shape) throw Error::tensorShapeMismatch("K and V caches must have one shape.");
        const int r = kc.shape.rank();
        if (r < 3 || (r == 4 && kc.shape[0] != 1) || r > 4) throw Error::tensorShapeMismatch("caches must be [1?, Nkv, Smax, Hd].");
        const int64_t Nkv = kc.shape[r - 3], Smax = kc.shape[r - 2], Hd = kc.shape[r - 1];
        if (kc.dataType != o || a.vCache->dataType != o || o != t)
            throw Error::unsupportedDataTypeCombination("KV scatter writes caches of the weight dtype.");
        if (a.position->dataType != DataType::i32) throw Error::unsupportedDataTypeCombination("position tensor must be i32");
        requireElements(*a.position, 1, "position");
        if (a.qRows < 0 || a.qRows + 2 * Nkv * Hd != N)
            throw Error::tensorShapeMismatch("weight rows must be qRows + 2 * Nkv * Hd for the KV scatter.");
        requireElements(*a.out, a.qRows, "DecodeMatvec out");
        flags |= 4u;
        dc.qRows = (uint32_t)a.qRows;
        dc.kvRows = (uint32_t)(Nkv * Hd);
        dc.headDim = (uint32_t)Hd;
        dc.kvStride = (uint32_t)Smax;
    } else {
        requireElements(*a.out, N, "DecodeMatvec out");
    }
    dc.flags = flags;
    const Tensor &x = *a.x;
    if (q4) {
        const AffineQuantizedTensor &Q = *a.qweight;
        const int lpr = q4Shape(N, K, false).lpr;
        const std::string fn = std::string("q4_decode_matvec_bf16_") + tag(o) + "_l" + std::to_string(lpr) + "_f" +
                               std::to_string(flags & 3u);
        AffineQMatmulConstants qc{1u, (uint32_t)N, (uint32_t)K, (uint32_t)(K / 64), (uint32_t)(K / 8), Q.hasBiases ? 1u : 0u};
        std::vector<Binding> b = {
            {x, kRead},
            {a.delta ? *a.delta : x, kRead},
            {a.wPost ? *a.wPost : x, kRead},
            {a.wPre ? *a.wPre : x, kRead},
            {Q.packedValues, kRead},
            {Q.scales, kRead},
            {Q.hasBiases ? Q.biases : Q.scales, kRead},
            {*a.out, kWrite},
            {a.xOut ? *a.xOut : x, a.xOut ? kWrite : kRead},
            {a.kCache ? *a.kCache : *a.out, kWrite},
            {a.vCache ? *a.vCache : *a.out, kWrite},
            {a.position ? *a.position : x, kRead},
        };
        // LDS: x as f32, its bf16 pair words (36 words per group of 64), the group sums
        const size_t lds = (size_t)K * 4 + (size_t)(K / 64) * 36 * 4 + (size_t)(K / 64) * 4;
        return std::make_unique<FixedDispatch>(fn, std::move(b), std::vector<std::vector<uint8_t>>{bytesOf(dc), bytesOf(qc)},
                                               grid1(streamBlocks(cdiv(N, 64 / lpr)), kBlock, lds));
    }
    const int R = matvecRows(N);
    const std::string fn = std::string("decode_matvec_") + tag(t) + "_" + tag(o) + "_r" + std::to_string(R) + "_f" +
                           std::to_string(flags & 3u);
    const Tensor &W = *a.weight;
    std::vector<Binding> b = {
        {x, kRead},
        {a.delta ? *a.delta : x, kRead},
        {a.wPost ? *a.wPost : x, kRead},
        {a.wPre ? *a.wPre : x, kRead},
        {W, kRead},
        {*a.out, kWrite},
        {a.xOut ? *a.xOut : x, a.xOut ? kWrite : kRead},
        {a.kCache ? *a.kCache : *a.out, kWrite},
        {a.vCache ? *a.vCache : *a.out, kWrite},
        {a.position ? *a.position : x, kRead},
    };
    return std::make_unique<FixedDispatch>(fn, std::move(b), std::vector<std::vector<uint8_t>>{bytesOf(dc)},
                                           grid1(streamBlocks(cdiv(N, R)), kBlock, (size_t)K * 4));
}

// EmbeddingGather.swift: ids [N] i32, table [V, H], out [N, H]
std::unique_ptr<Kernel> EmbeddingGather(const Tensor &ids, const Tensor &table, const Tensor &out) {
    using D = DataType;
    if (ids.dataType != D::i32) throw Error::unsupportedDataTypeCombination("EmbeddingGather ids must be i32.");
    if (table.shape.rank() != 2) throw Error::tensorInvalidRank(2, table.shape.rank());
    const int64_t V = table.shape[0], H = table.shape[1], N = ids.shape.elementCount();
    const char *fn = nullptr;
    if (table.dataType == D::f32 && out.dataType == D::f32) fn = "embedding_gather";
    else if (table.dataType == D::f16 && out.dataType == D::f16) fn = "embedding_gather_f16";
    else if (table.dataType == D::bf16 && out.dataType == D::bf16) fn = "embedding_gather_bf16";
    else if (table.dataType == D::bf16 && out.dataType == D::f32) fn = "embedding_gather_bf16_to_f32";
    else throw Error::unsupportedDataTypeCombination("Unsupported EmbeddingGather data type combination.");
    requireElements(out, N * H, "EmbeddingGather out");
    EmbeddingGatherExtConstants ec{(uint32_t)N, (uint32_t)H, (uint32_t)V};
    const int64_t runs = N * cdiv(H, 16 / stride(table.dataType));
    return std::make_unique<FixedDispatch>(std::string(fn) + "_ext",
                                           std::vector<Binding>{{ids, kRead}, {table, kRead}, {out, kWrite}},
                                           std::vector<std::vector<uint8_t>>{bytesOf(ec)},
                                           grid1(runs ? std::clamp<int64_t>(cdiv(runs, kBlock), 1, 4096) : 0, kBlock));
}


// The 4-bit Matmul on the matrix cores for bf16 rows (aq_gemm.hip): x's
// group sums and a pair-ordered copy of x in scratch, then 128 x 128 tiles
// of C, with the K groups split over blocks (and a reduction) when the tiles
// leave CUs idle. Its three launches take ~25-35 us at small m, while the
// streaming matvec per row costs about N K / 2 bytes / 4.5 TB/s per row, so
// the GEMM wins once the rows' weight reads pass ~2^27 bytes (measured at
// N K = 9216 x 2304 both ways: 26 against 43 us at m 16-29, 35 against
// 210 us at m 128).
constexpr int64_t kQ4GemmMinRows = 16;
constexpr int64_t kQ4GemmMinBytes = int64_t{1} << 27;  // m * N * K / 2

class AffineQGemmKernel : public Kernel {
public:
    AffineQGemmKernel(const Tensor &a, const AffineQuantizedTensor &b, const Tensor &c, const AffineQMatmulConstants &qc)
        : a_(a), b_(b), c_(c), qc_(qc) {}
    std::vector<Binding> tensors() const override {
        std::vector<Binding> t = {{b_.packedValues, kRead}, {b_.scales, kRead}, {a_, kRead}, {c_, kWrite}};
        if (b_.hasBiases) t.push_back({b_.biases, kRead});
        return t;
    }
    std::string describe() const override {
        return "aq_gemm_prep_bf16," + mainName() + (splits() > 1 ? "," + reduceName() : std::string());
    }
    void encode(KernelCommandEncoder &enc) const override {
        const int64_t m = qc_.M, k = qc_.K, g = qc_.kGroups, n = qc_.N, tiles = cdiv(m, 128) * cdiv(n, 128);
        const int64_t s = splits();
        enc.withTemporaryTensor(ScratchSpec{{m, k}, DataType::bf16}, [&](Tensor xp) {
            enc.withTemporaryTensor(ScratchSpec{{m, g}, DataType::f32}, [&](Tensor xs) {
                FixedDispatch prep("aq_gemm_prep_bf16", {{a_, kRead}, {xp, kWrite}, {xs, kWrite}}, {bytesOf(qc_)},
                                   grid1(cdiv(m * (k / 8), kBlock), kBlock));
                enc.dispatch(prep);
                const Tensor &bias = b_.hasBiases ? b_.biases : b_.scales;
                if (s <= 1) {
                    FixedDispatch gemm(mainName(),
                                       {{b_.packedValues, kRead}, {b_.scales, kRead}, {bias, kRead}, {xp, kRead},
                                        {xs, kRead}, {c_, kWrite}},
                                       {bytesOf(qc_)}, grid1(tiles, kBlock));
                    enc.dispatch(gemm);
                    return;
                }
                enc.withTemporaryTensor(ScratchSpec{{s * m, n}, DataType::f32}, [&](Tensor part) {
                    DispatchSize ds;
                    ds.grid = dim3((unsigned)tiles, (unsigned)s, 1);
                    ds.block = dim3(kBlock, 1, 1);
                    FixedDispatch gemm(mainName(),
                                       {{b_.packedValues, kRead}, {b_.scales, kRead}, {bias, kRead}, {xp, kRead},
                                        {xs, kRead}, {part, kWrite}},
                                       {bytesOf(qc_)}, ds);
                    enc.dispatch(gemm);
                    MatmulConstants mc{(uint32_t)m, (uint32_t)k, (uint32_t)n, 1u};
                    const uint32_t splits = (uint32_t)s;
                    const int64_t blocks = std::clamp<int64_t>(cdiv(m * n / 4, kBlock), 1, 8 * deviceCUs());
                    FixedDispatch reduce(reduceName(), {{part, kRead}, {c_, kWrite}}, {bytesOf(mc), bytesOf(splits)},
                                         grid1(blocks, kBlock));
                    enc.dispatch(reduce);
                });
            });
        });
    }

private:
    // K splits (groups per block) when the tiles leave CUs idle: about two
    // blocks per CU, at least 4 groups each; the reduction takes M N % 4 == 0
    // and 16-byte-aligned C
    int64_t splits() const {
        const int64_t tiles = cdiv((int64_t)qc_.M, 128) * cdiv((int64_t)qc_.N, 128);
        const int64_t want = 2 * (int64_t)deviceCUs() / std::max<int64_t>(tiles, 1);
        const int64_t s = std::min<int64_t>(want, (int64_t)qc_.kGroups / 4);
        const bool reducible = ((int64_t)qc_.M * qc_.N) % 4 == 0 && aligned16(c_.data);
        return reducible && s >= 2 ? s : 1;
    }
    // Waves of 64 x 64 where all blocks run in one round of two per CU with more
    // than 36 groups each, else of 128 x 32 (aq_gemm.hip). Over 260 shapes, 128 x
    // 32 against 64 x 64: up to 36 groups 2.3% faster (2 of 97 over 2% slower, the
    // worst 4%), more blocks 5% faster (none over 2% slower), the rest equal on
    // average with 45 of 127 over 2% slower, the worst 10%.
    std::string mainName() const {
        const int64_t s = splits(), blocks = cdiv((int64_t)qc_.M, 128) * cdiv((int64_t)qc_.N, 128) * s;
        const bool w64 = blocks <= 2 * (int64_t)deviceCUs() && cdiv((int64_t)qc_.kGroups, s) > 36;
        return std::string("aq_gemm_mfma_bf16_bf16_") + (s > 1 ? "splitk" : tag(c_.dataType)) + "_b4_g64" + (w64 ? "_w64" : "");
    }
    std::string reduceName() const { return std::string("matmul_splitk_reduce_") + tag(c_.dataType); }
    Tensor a_;
    AffineQuantizedTensor b_;
    Tensor c_;
    AffineQMatmulConstants qc_;
};

// A few bf16 rows through a 4-bit matrix (aq_rows.hip): the row tiles of 16,
// the waves that share a tile's K, and the values of K staged per phase.
struct AqRowsPlan {
    int mt = 0, wk = 1;  // mt 0: not this kernel
    int64_t kp = 0;
    size_t lds = 0;
};

AqRowsPlan aqRowsPlan(int64_t m, int64_t n, int64_t k) {
    AqRowsPlan r;
    // Against one matvec per row (m < 16, or under 2^27 weight bytes in all),
    // whose time grows with m n k while this kernel's fixed cost is 5-6 us:
    // from 25 million multiply-adds on (K 2304, N 2304: m 4 6.2 against 6.3 us,
    // m 8 8.4 against 6.5), two rows from 2^26 (K 2304, N 9216: 9.1 against
    // 9.9; K 3072, N 24576: 20.6 against 17.7), and not below 1024 rows of W
    // (K 8192, N 500, m 8: 8.1 against 11.5).
    if (m < 2 || m > 64 || n < 1024 || m * n * k < (m == 2 ? int64_t{1} << 26 : 25000000)) return r;
    // Against the prompt GEMM (aq_gemm.hip): up to 48 rows, while x fits one or
    // two phases (K 2304, N 9216, m 16: 22.1 against 10.9 us, m 48 27.1 against
    // 22.8; K 9216, N 2304, m 24 28.8 against 23.8, m 32 29.8 against 30.9).
    // K under 2048 stays there too: the routing tests hold it (K 1024, N 16448,
    // m 16: 19.5 against 7.6).
    if (m >= kQ4GemmMinRows && m * n * (k / 2) >= kQ4GemmMinBytes && (k < 2048 || m > 48)) return r;
    if (m >= kQ4GemmMinRows && m * k > (m <= 32 ? 230000 : 165000)) return r;
    r.mt = m <= 16 ? 1 : m <= 32 ? 2 : 4;
    // the fewest waves per tile (x is staged once per block) that give more
    // blocks than half the CUs: N 9216 144 blocks of 4 tiles (288 of 2 tiles:
    // 11.3 us), N 4096 256 blocks of one (128 of two: 8.1 against 7.0)
    while (r.wk < 8 && cdiv(n, 16 * (8 / r.wk)) * 2 <= deviceCUs()) r.wk *= 2;
    // x and its group sums in up to 152 KB of LDS, in equal phases
    auto bytes = [&](int64_t kp) { return (size_t)(m * (kp * 2 + 16) + kp / 64 * 16 * r.mt * 4); };
    for (int64_t phases = 1;; ++phases) {
        r.kp = cdiv(k / 128, phases) * 128;
        if (bytes(r.kp) <= 152 * 1024 || r.kp == 128) break;
    }
    r.lds = std::max(bytes(r.kp), (size_t)(8 * r.mt * 1024));  // the waves' sums take its place at the end
    return r;
}

// Matmul.swift:99-130 and :279-332
std::unique_ptr<Kernel> Matmul(const Tensor &a, const AffineQuantizedTensor &b, const Tensor &c) {
    using D = DataType;
    b.validate();
    if (a.shape.rank() != 2) throw Error::tensorInvalidRank(2, a.shape.rank());
    if (c.shape.rank() != 2) throw Error::tensorInvalidRank(2, c.shape.rank());
    const int64_t m = a.shape[0], k = a.shape[1], n = b.outFeatures();
    if (b.inFeatures() != k)
        throw Error::tensorShapeMismatch("Matmul quantized RHS shape mismatch: a.shape=[" + std::to_string(m) + "," +
                                         std::to_string(k) + "] but b.inFeatures=" + std::to_string(b.inFeatures()) + ".");
    if (c.shape != Shape{m, n})
        throw Error::tensorShapeMismatch("Matmul output shape mismatch: expected [" + std::to_string(m) + "," + std::to_string(n) +
                                         "], got " + c.shape.str() + ".");
    if (b.groupSize <= 0 || k % b.groupSize != 0)
        throw Error::tensorShapeMismatch("Matmul quantized RHS: K=" + std::to_string(k) + " is not divisible by groupSize=" +
                                         std::to_string(b.groupSize) + ".");
    const D x = a.dataType, sd = b.scales.dataType, o = c.dataType;
    const bool combo = (x == D::bf16 && sd == D::bf16 && (o == D::bf16 || o == D::f32)) ||
                       (x == D::f32 && sd == D::bf16 && o == D::f32);
    if (b.bits != 4 || b.groupSize != 64 || !combo)
        throw Error::unsupportedDataTypeCombination(
            "Unsupported affine quantized matmul combination: format=(bits: " + std::to_string(b.bits) + ", groupSize: " +
            std::to_string(b.groupSize) + "), x=" + tag(x) + ", scales=" + tag(sd) + ", out=" + tag(o) + ".");
    if (m > UINT32_MAX || n > UINT32_MAX || k > UINT32_MAX) throw Error::tensorShapeMismatch("Matmul dimensions out of range.");
    requireElements(a, m * k, "Matmul a");
    requireElements(c, m * n, "Matmul c");
    requireElements(b.packedValues, n * (k / 8), "Matmul quantized packed values");
    requireElements(b.scales, n * (k / 64), "Matmul quantized scales");
    if (b.hasBiases) requireElements(b.biases, n * (k / 64), "Matmul quantized biases");
    AffineQMatmulConstants qc{(uint32_t)m, (uint32_t)n, (uint32_t)k, (uint32_t)(k / 64), (uint32_t)(k / 8), b.hasBiases ? 1u : 0u};
    const Tensor &bias = b.hasBiases ? b.biases : b.scales;
    std::vector<Binding> binds = {{b.packedValues, kRead}, {b.scales, kRead}, {bias, kRead}, {a, kRead}, {c, kWrite}};
    const std::string combo3 = std::string(tag(x)) + "_bf16_" + tag(o) + "_b4_g64";
    const Q4Shape q = q4Shape(n, k, x == D::f32);
    const bool aligned = aligned16(b.packedValues.data) && aligned16(a.data) &&
                         (reinterpret_cast<uintptr_t>(b.scales.data) & 3) == 0 && (reinterpret_cast<uintptr_t>(bias.data) & 3) == 0;
    const int64_t lim = int64_t{1} << 31;
    if (x == D::bf16 && o == D::bf16 && aligned && k % 128 == 0 && n * (k / 2) < lim && m * k * 2 < lim) {
        const AqRowsPlan r = aqRowsPlan(m, n, k);
        if (r.mt) {
            const uint32_t kp = (uint32_t)r.kp;
            return std::make_unique<FixedDispatch>(
                "aq_matvec_simd4_" + combo3 + "_m" + std::to_string(r.mt) + "_s" + std::to_string(r.wk), binds,
                std::vector<std::vector<uint8_t>>{bytesOf(qc), bytesOf(kp)}, grid1(cdiv(n, 16 * (8 / r.wk)), 512, r.lds));
        }
    }
    // a prompt's rows of bf16 activations: the matrix-core GEMM (one pass
    // over the weights for all rows instead of one matvec per row)
    // (buffer copies: every operand under 2^31 bytes; an even number of
    // groups per row, so a group's scale and bias share a 32-bit word with
    // a neighbour of the same row)
    if (x == D::bf16 && m >= kQ4GemmMinRows && m * n * (k / 2) >= kQ4GemmMinBytes && aligned && k % 128 == 0 &&
        m * k * 2 < lim && n * (k / 2) < lim && m * (k / 64) * 4 < lim && cdiv(m, 128) * cdiv(n, 128) <= (int64_t)UINT32_MAX)
        return std::make_unique<AffineQGemmKernel>(a, b, c, qc);
    DispatchSize ds;
    ds.block = dim3(kBlock, 1, 1);
    std::string fn;
    if (q.lpr && aligned && m <= 65535) {
        fn = std::string(m == 1 ? "aq_qmv_fast_" : "aq_matvec_simd4_") + combo3 + "_l" + std::to_string(q.lpr) + "_j" +
             std::to_string(q.j);
        const int64_t units = cdiv(n, 64 / q.lpr);
        ds.grid = dim3((unsigned)streamBlocks(units), (unsigned)m, 1);
    } else {
        if (m > 65535) throw Error::tensorShapeMismatch("quantized Matmul supports at most 65535 rows of a.");
        // the reference's kernel: a 32-lane half-wave per 4 rows, 8 per block
        fn = "aq_matvec_simd4_" + combo3;
        ds.grid = dim3((unsigned)cdiv(cdiv(n, 4), kBlock / 32), (unsigned)m, 1);
    }
    if (m == 0 || n == 0) ds.grid = dim3(0, 1, 1);
    return std::make_unique<FixedDispatch>(fn, binds, std::vector<std::vector<uint8_t>>{bytesOf(qc)}, ds);
}

// EmbeddingGather.swift:45-88
std::unique_ptr<Kernel> EmbeddingGather(const Tensor &ids, const AffineQuantizedTensor &table, const Tensor &out) {
    using D = DataType;
    table.validate();
    if (ids.shape.rank() != 1) throw Error::tensorInvalidRank(1, ids.shape.rank());
    if (ids.dataType != D::i32)
        throw Error::unsupportedDataTypeCombination(std::string("EmbeddingGather with quantized table requires i32 ids; got ") +
                                                    tag(ids.dataType) + ".");
    if (out.shape.rank() != 2) throw Error::tensorInvalidRank(2, out.shape.rank());
    const int64_t T = ids.shape[0], H = table.inFeatures(), V = table.outFeatures();
    if (out.shape != Shape{T, H})
        throw Error::tensorShapeMismatch("EmbeddingGather output shape mismatch: expected [" + std::to_string(T) + "," +
                                         std::to_string(H) + "], got " + out.shape.str() + ".");
    if (table.groupSize <= 0 || H % table.groupSize != 0)
        throw Error::tensorShapeMismatch("EmbeddingGather quantized table hiddenSize=" + std::to_string(H) +
                                         " is not divisible by groupSize=" + std::to_string(table.groupSize) + ".");
    if (table.bits != 4 || table.groupSize != 64)
        throw Error::unsupportedDataTypeCombination(
            "EmbeddingGather currently only supports affine quantized tables with bits=4, groupSize=64, "
            "packing=.uint32LittleEndian.");
    if (table.scales.dataType != D::bf16 || !(out.dataType == D::bf16 || out.dataType == D::f32))
        throw Error::unsupportedDataTypeCombination(std::string("Unsupported quantized EmbeddingGather combination: scales ") +
                                                    tag(table.scales.dataType) + ", out " + tag(out.dataType) + ".");
    if (V > UINT32_MAX || H > UINT32_MAX || T > UINT32_MAX) throw Error::tensorShapeMismatch("EmbeddingGather dimensions out of range.");
    requireElements(table.packedValues, V * (H / 8), "EmbeddingGather quantized packed values");
    requireElements(table.scales, V * (H / 64), "EmbeddingGather quantized scales");
    if (table.hasBiases) requireElements(table.biases, V * (H / 64), "EmbeddingGather quantized biases");
    requireElements(out, T * H, "EmbeddingGather out");
    AffineQEmbeddingGatherExtConstants gc{(uint32_t)T, (uint32_t)H, (uint32_t)(H / 64), (uint32_t)(H / 8),
                                          table.hasBiases ? 1u : 0u, (uint32_t)V};
    const Tensor &bias = table.hasBiases ? table.biases : table.scales;
    const std::string fn = std::string("aq_embedding_gather_bf16_") + tag(out.dataType) + "_b4_g64_ext";
    const int64_t words = T * (H / 8);
    return std::make_unique<FixedDispatch>(
        fn, std::vector<Binding>{{ids, kRead}, {table.packedValues, kRead}, {table.scales, kRead}, {bias, kRead}, {out, kWrite}},
        std::vector<std::vector<uint8_t>>{bytesOf(gc)}, grid1(words ? std::clamp<int64_t>(cdiv(words, kBlock), 1, 4096) : 0, kBlock));
}

// Argmax.swift:24-37
std::unique_ptr<Kernel> Argmax(const Tensor &x, const Tensor &indices) {
    const int rank = x.shape.rank();
    if (rank <= 0) throw Error::tensorInvalidAxis(-1, rank);
    const int64_t n = x.shape[rank - 1];
    const int64_t rows = n ? x.shape.elementCount() / n : 0;
    if (indices.shape.elementCount() != rows)
        throw Error::tensorShapeMismatch("Argmax indices must contain " + std::to_string(rows) + " elements; got " +
                                         std::to_string(indices.shape.elementCount()) + ".");
    return std::make_unique<ArgmaxKernel>(x, indices, rows, n);
}

std::unique_ptr<Kernel> Custom(const std::string &functionName, std::vector<Binding> tensors,
                               std::vector<std::vector<uint8_t>> constants, dim3 grid, dim3 block) {
    return Custom(functionName, std::move(tensors), std::move(constants), grid, block, 0);
}

std::unique_ptr<Kernel> Custom(const std::string &functionName, std::vector<Binding> tensors,
                               std::vector<std::vector<uint8_t>> constants, dim3 grid, dim3 block, size_t dynamicLds) {
    DispatchSize ds;
    ds.grid = grid;
    ds.block = block;
    ds.dynamicLds = dynamicLds;
    return std::make_unique<FixedDispatch>(functionName, std::move(tensors), std::move(constants), ds);
}

std::unique_ptr<Kernel> FillNormal(void *data, DataType dtype, uint64_t count, uint64_t seed, float mean, float stddev) {
    if (!isFloat(dtype)) throw Error::unsupportedDataTypeCombination("fill_normal writes f32, f16 or bf16.");
    if (count && !data) throw Error::invalidArgument("fill_normal: null data pointer");
    FillNormalConstants fc{seed, count, mean, stddev};
    Tensor t(data, Shape({(int64_t)count}), dtype);
    const int64_t blocks = std::clamp<int64_t>(cdiv((int64_t)count, kBlock), 1, 16 * deviceCUs());
    return std::make_unique<FixedDispatch>(std::string("fill_normal_") + tag(dtype), std::vector<Binding>{{t, kWrite}},
                                           std::vector<std::vector<uint8_t>>{bytesOf(fc)}, grid1(count ? blocks : 0, kBlock));
}

}  // namespace Kernels
}  // namespace popcorn

// ---------------------------------------------------------------------------
// The merged-pair exchange of the tiled prefill attention, per stream
// ---------------------------------------------------------------------------

namespace popcorn {
namespace {

struct PairExchangeRegistry {
    std::mutex mu;
    std::map<std::pair<int, hipStream_t>, PairExchange> byStream;
};
PairExchangeRegistry &pairRegistry() {
    static auto *r = new PairExchangeRegistry();  // lives to process exit, as the memory does
    return *r;
}

size_t roundUpPow2(size_t n) {
    size_t p = 1 << 20;
    while (p < n) p <<= 1;
    return p;
}

// Reads the abort word; when set, clears every flag and throws -1019.
void checkOne(const PairExchange &x) {
    uint64_t abortWord = 0;
    checkHip(hipMemcpy(&abortWord, x.flags, 8, hipMemcpyDeviceToHost), "read the pair exchange's abort word");
    if (abortWord == 0) return;
    checkHip(hipMemset(x.flags, 0, PairExchange::kFlags * 8), "clear the pair exchange's flags");
    throw Error(POPCORN_ERR_GPU_INTERNAL,
                "FlashAttention: a merged causal tile pair's ready-flag wait gave up (0.2 s, or a flag left by a "
                "launch that gave up before); the affected output rows hold NaN. The flags have been cleared.");
}

}  // namespace

PairExchange &pairExchange(hipStream_t stream, size_t dataBytes) {
    int dev = 0;
    checkHip(hipGetDevice(&dev), "hipGetDevice");
    auto &r = pairRegistry();
    std::lock_guard<std::mutex> g(r.mu);
    PairExchange &x = r.byStream[{dev, stream}];
    if (!x.flags) {
        x.flags = static_cast<uint64_t *>(UncachedPool::take(PairExchange::kFlags * 8));
        x.dev = dev;
        checkHip(hipMemset(x.flags, 0, PairExchange::kFlags * 8), "zero the pair exchange's flags");
    }
    if (x.dataBytes < dataBytes) {
        // the old block stays reserved: a graph captured with it still uses it
        const size_t n = roundUpPow2(dataBytes);
        x.data = UncachedPool::take(n);
        x.dataBytes = n;
    }
    return x;
}

bool pairExchangeHeld(hipStream_t stream, size_t dataBytes) {
    int dev = 0;
    checkHip(hipGetDevice(&dev), "hipGetDevice");
    auto &r = pairRegistry();
    std::lock_guard<std::mutex> g(r.mu);
    const auto it = r.byStream.find({dev, stream});
    return it != r.byStream.end() && it->second.flags && it->second.dataBytes >= dataBytes;
}

void checkPairExchange(hipStream_t stream, bool allStreams) {
    int dev = 0;
    checkHip(hipGetDevice(&dev), "hipGetDevice");
    auto &r = pairRegistry();
    std::vector<PairExchange> todo;
    {
        std::lock_guard<std::mutex> g(r.mu);
        for (auto &kv : r.byStream)
            if (kv.first.first == dev && (allStreams || kv.first.second == stream)) todo.push_back(kv.second);
    }
    for (const PairExchange &x : todo) checkOne(x);
}

}  // namespace popcorn
