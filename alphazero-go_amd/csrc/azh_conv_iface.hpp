// The 3x3 convolutions' interface (the stem's, azh_conv.hpp, and the
// residual tower's, azh_tower.hpp): weight packing, workgroup shapes, the
// launchers and the BN/skip/ReLU epilogue. Kept apart from the other
// kernels' declarations so that a hash of the convolutions' sources changes
// only with them.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace azh {

// Channels per K chunk of the stem's convolution: 4 groups of 4 channels.
constexpr int kChunk = 16;
// Channels per K chunk of the tower's: 4 groups of 8 channels.
constexpr int kTowerChunk = 32;
// Output channels per MFMA block (16 x 16 outputs).
constexpr int kCoBlock = 16;

inline int ceilDiv(int a, int b) { return (a + b - 1) / b; }

// Output-channel blocks of packed weights: ceil(cout/16) rounded up to whole
// 128-channel workgroup tiles, so no workgroup shape reads past them.
inline int packedCoBlocks(int cout) { return ceilDiv(ceilDiv(cout, kCoBlock), 8) * 8; }

// The stem's weights w [cout][cin][3][3] (Conv2d::w,
// include/azgo/layers.hpp:32, row (c*3 + dy)*3 + dx) packed as the MFMA A
// fragments the kernel loads: [co block][chunk q][tap t][lane 0..63][j 0..3],
// value w[cb*16 + (lane & 15)][q*16 + 4*(lane >> 4) + j][t], zero where the
// output or input channel is padding. co blocks = packedCoBlocks(cout),
// chunks = ceil(cin/16).
std::vector<float> packConv3x3(const float* w, int cin, int cout);
size_t packedConv3x3Floats(int cin, int cout);

// A tower layer's weights on the device.
// parts: the weights w [cout][cin][3][3] split in two f16 parts
// (azh_tower.hpp), w * 2^wexp[co] = h + l, the power of two taking the
// channel's largest finite weight into [2^14, 2^15), packed as the MFMA A
// fragments the kernel loads: [co block][chunk q][tap t][part h, l][lane
// 0..63][j 0..7], value w[cb*16 + (lane & 15)][q*32 + 8*(lane >> 4) + j][t],
// zero where the channel is padding (co blocks = packedCoBlocks(cout), chunks
// = ceil(cin/32); but the output channels that fill up the last quad repeat
// its last one) or the weight an infinity or a NaN.
// wexp: cout powers of two.
// least: per channel, the magnitude a sum of the parts' products (that is,
// 2^wexp and the activations' power of two in it) has to reach for what the
// parts miss to be lost in its rounding (azh_tower.hpp); infinite for a
// channel with an infinity or a NaN among its weights.
// rest: of the weights that the parts miss by more than 2^-23 of them (2^-16
// and less of the channel's largest), the difference: kRests a channel, in
// the order of their index c * 9 + t, -1 after the last. A layer with more in
// a channel, or an infinity or a NaN, needs w.
// w: the weights as given, for the outputs that the split cannot give; null
// in a network that parts and rests hold.
struct WeightRest {
    int index;
    float value;
};
constexpr int kRests = 8;
struct TowerWeights {
    const float* parts;
    const int* wexp;
    const float* least;
    const float* scale;   // folded BN
    const float* shift;
    const WeightRest* rest;
    const float* w;
};
// Layers of such weights, one after the other `stride` words apart, each
// array but w at its offset in the layer's.
struct TowerLayers {
    float* base;
    const float* w;
    size_t stride, wStride;
    unsigned scale, shift, wexp, least, rest, parts;   // 32 bits: an address costs the kernels fewer scalar registers
    __host__ __device__ TowerWeights at(int l) const {
        const float* p = base + (size_t)l * stride;
        return {p + parts,
                reinterpret_cast<const int*>(p + wexp),
                p + least,
                p + scale,
                p + shift,
                reinterpret_cast<const WeightRest*>(p + rest),
                w ? w + (size_t)l * wStride : nullptr};
    }
};
// The offsets and strides of a layer (base and w null): every array starts and
// ends at a multiple of 64 words, the first four are zeros past cout.
TowerLayers towerLayers(int cin, int cout);
// Fills parts, wexp, least and rest of `layers` layers from layer `first` on, from
// their weights w (one after the other) on the device. Sets *needsW where a
// layer needs its weights as given.
hipError_t launchPackTower(const TowerLayers& t, int first, int layers, const float* w, int cin, int cout, int* needsW,
                           hipStream_t stream);

// How a convolution launch is cut: output channels per workgroup (a
// multiple of 16) and the resulting number of co tiles. The cut only
// decides which workgroup computes an output, never how: every output
// channel sums its inputs in one fixed order (the tower's: chunk, tap, the
// parts' products l, h, then h, l last, azh_tower.hpp; the stem's: chunk,
// tap, channel in chunk, its short last chunk of input planes in the packed
// (plane, tap) order of azh_stem.hpp), so results are bitwise independent of
// the cut and of the batch.
struct ConvTiling {
    int coPerWave;   // MFMA blocks of 16 output channels per wave: 1 or 2
    int wavesCo;     // waves along the output channels (at most 128 channels per workgroup)
    int wavesPg;     // waves along the board's 16-point column groups
    int pgPerWave;   // column groups per wave; 0: all of the board's
    int waves() const { return wavesCo * wavesPg; }
    int coTile() const { return 16 * coPerWave * wavesCo; }
};
// The tower's shape for a pass over B boards in all. alone: no other pass is
// in flight on the device (the runner's other slots idle), which admits the
// shapes that are fastest for one pass but slower for two side by side.
ConvTiling chooseTowerTiling(int cout, int B, int boardSize, bool alone = false);
// The stem's.
ConvTiling chooseStemTiling(int cout, int B, int boardSize, bool alone = false);
inline constexpr bool operator==(const ConvTiling& a, const ConvTiling& b) {
    return a.coPerWave == b.coPerWave && a.wavesCo == b.wavesCo && a.wavesPg == b.wavesPg &&
           a.pgPerWave == b.pgPerWave;
}

// The workgroup shapes the stem's convolution is built for, in the order a
// probe indexes them. Each is compiled for every supported board size.
constexpr ConvTiling kConvTilings[] = {{2, 2, 2, 12}, {1, 4, 1, 0}, {1, 2, 1, 0}, {1, 1, 1, 0}, {1, 8, 1, 0},
                                       {1, 2, 2, 12}, {1, 1, 4, 6}, {1, 1, 4, 2}, {1, 1, 4, 1}, {1, 1, 8, 1},
                                       {1, 1, 3, 1}, {1, 1, 6, 1}, {1, 1, 6, 2}};
constexpr int kConvTilingCount = sizeof kConvTilings / sizeof kConvTilings[0];
// The tower's (as many, so that a probe's index names one of either).
constexpr ConvTiling kTowerTilings[] = {{2, 4, 2, 0}, {2, 2, 4, 0}, {2, 1, 4, 0}, {1, 1, 4, 0}, {2, 2, 2, 0},
                                        {2, 2, 4, 3}, {2, 1, 4, 3}, {1, 2, 4, 3}, {1, 2, 3, 2}, {1, 1, 3, 2},
                                        {1, 1, 1, 1}, {1, 1, 3, 1}, {1, 2, 3, 1}};
static_assert(sizeof kTowerTilings / sizeof kTowerTilings[0] == kConvTilingCount, "one index for either list");
// The tower kernel's compile-time settings of a shape: the waves per SIMD
// its registers are budgeted for, and how many taps' A fragments a wave
// keeps in registers (all but one of them in flight). Small pixel tiles take
// nine: their taps are three MFMAs or few more, far shorter than a load.
// (Two or four chunks' fragments ahead measured slower, 8.8 against 7.3 us a
// layer of one 19x19 board at 128 channels: the waves of a tile fetch the
// same fragments, and the CU's vector memory path is what they wait for.)
constexpr int towerWavesPerSimd(int threads) { return threads >= 512 ? 2 : 1; }
constexpr int towerTapRing(int coPerWave, int pgPerWave) { return coPerWave == 1 && pgPerWave != 0 ? 9 : 3; }
// LDS cells (16 bytes) of one 8-channel group of `rows` staged rows and two
// halo rows of n + 1, and the last row's right halo, rounded up to 16: the
// lanes that one phase of a ds_read_b128 serves come from two channel groups,
// which then fall in different banks. At 441 cells (rows of n + 2, 19x19) the
// board-resident tower lost 125.6 M LDS cycles to bank conflicts, at 432 64.5
// M; a layer of 256 channels over 16 19x19 boards in the shape {1, 2, 3, 2}
// took 35.8 us, now 31.1, one of 128 channels over 8 11.2, now 10.1.
constexpr int towerGroupCells(int rows, int n) { return ((rows + 2) * (n + 1) + 1 + 15) / 16 * 16; }
// The smallest shapes (azh_tower.hpp, towerDeep): threads of a workgroup, and
// chunks of K staged at once.
constexpr int kDeepThreads = 512, kDeepChunks = 4;
constexpr bool towerDeepShape(int wavesCo, int wavesPg, int pgPerWave) {
    return wavesCo == 1 && wavesPg <= 3 && pgPerWave == 1;
}

// Trunk activations (every convolution's output, the residual input and the
// tower's input) are stored in channel quads: [B][ceil(C/4)][n*n][4], the
// four channels 4g..4g+3 of a point side by side. A lane then moves four
// channels with one 16-byte access: the LDS staging wants exactly that
// interleave, and an MFMA lane's accumulators are four consecutive channels
// of one point. Channels past C in the last quad are stored as zeros. The
// network's input planes stay [B][P][n*n], as the reference hands them over.
inline int channelQuads(int channels) { return ceilDiv(channels, 4); }
inline size_t quadFloats(int B, int channels, int points) { return (size_t)B * channelQuads(channels) * 4 * points; }

// Reorders between the planar [B][C][A] layout and channel quads (zeros in
// the padding), on the host: for test hooks that take or return planar data.
std::vector<float> toChannelQuads(const float* planar, int B, int C, int A);
void fromChannelQuads(const float* quads, int B, int C, int A, float* planar);

// A convolution hands the next one each board's largest magnitude, which
// its operands' scale is made from (azh_tower.hpp): every wave writes the
// biased exponent of its own outputs' largest (255: an infinity or a NaN; 0:
// nothing but zeros) to one byte, board b's wave i at bytes + b * stride + i.
struct BoardScales {
    const uint8_t* in;   // the input boards' (tower): inParts bytes each
    uint8_t* out;        // this layer's (null: not reported): convParts(shape) each
    int inParts, stride;
};
// The waves of a shape that share a board: the bytes it reports per board.
int convParts(ConvTiling t, int cout, int boardSize);
// The same byte (one per board) for activations x [B][ceil(C/4)][n*n][4]
// that no convolution reported: one workgroup per board.
hipError_t launchBoardScales(const float* x, int B, int channels, int points, uint8_t* out, int stride,
                             hipStream_t stream);

// One (board size, workgroup shape) instance of the stem's convolution
// (azh_conv.hpp) and of the tower's (azh_tower.hpp; CH: for one or two chunks
// of input channels, 0: for more), instantiated by azh_conv_inst.hip, one
// object per shape and CH.
template <int N, int COW, int WCO, int WPG, int PPW>
hipError_t launchStemT(const float* x, const float* wp, const float* scale, const float* shift, const float* skip,
                       float* y, const BoardScales& s, int B, int cin, int cout, bool relu, hipStream_t stream);
template <int N, int COW, int WCO, int WPG, int PPW, int CH>
hipError_t launchTowerT(const float* x, const TowerWeights& w, const float* skip, float* y, const BoardScales& s, int B,
                        int cin, int cout, bool relu, hipStream_t stream);

// y[b][co][p] = relu?( (scale[co] * conv(x)[b][co][p] + shift[co]) (+ skip[b][co][p]) )
// with each multiply and add rounded separately (BatchNorm2d::forwardInfer,
// src/layers.cpp:88-97, then the skip add and reluForward,
// src/network.cpp:264-271). skip may alias y (in-place residual).
// y and skip in channel quads. The stem: x the network's input planes
// [B][cin][n*n], weights as packConv3x3 packs them; the tower: x a trunk
// activation in channel quads.
hipError_t launchStem(const float* x, const float* wPacked, const float* scale, const float* shift, const float* skip,
                      float* y, const BoardScales& s, int B, int n, int cin, int cout, bool relu, ConvTiling tiling,
                      hipStream_t stream);
hipError_t launchTower(const float* x, const TowerWeights& w, const float* skip, float* y, const BoardScales& s, int B,
                       int n, int cin, int cout, bool relu, ConvTiling tiling, hipStream_t stream);
bool conv3x3Supported(int boardSize);

// The stem and the residual tower in one launch, each board resident in one
// workgroup of 8 waves (128 output channels) from its first layer to its
// last (azh_resident.hpp): the per-layer launches' arithmetic without their
// kernel boundaries. For networks of 113-128 channels and stems of up to 32
// planes, on the board sizes residentTowerSupported names.
struct ResidentTower {
    const float* in;   // the network's input planes [B][P][A]; null: no stem (x holds the tower's input)
    const float *stemW, *stemScale, *stemShift;   // the stem's packed weights and folded BN
    int P;
    float* x;     // the trunk (channel quads), in place
    float* mid;   // the blocks' middle activations
    TowerLayers w;   // the tower's layers: conv1, conv2 of each block in turn
    int layers, B, F;
};
bool residentTowerSupported(int boardSize, int F, int P);
// workgroups: at most B; each takes every workgroups-th board.
hipError_t launchResidentTower(const ResidentTower& t, int boardSize, int workgroups, hipStream_t stream);
template <int N>
hipError_t launchResidentTowerT(const ResidentTower& t, int workgroups, hipStream_t stream);

// y = relu?(scale * acc + shift (+ skip)), each operation rounded on its own.
__device__ inline float epilogue(float acc, float s, float h, bool addSkip, float skipv, bool relu) {
    float v = __fadd_rn(__fmul_rn(s, acc), h);
    if (addSkip) v = __fadd_rn(v, skipv);
    if (relu) v = v > 0.0f ? v : 0.0f;   // -0 and NaN become +0 (reluForward)
    return v;
}

} // namespace azh
