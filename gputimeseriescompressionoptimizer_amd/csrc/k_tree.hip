// Device-side parse of a serialized compression tree (reference
// DecompressNodes, tree/compression_tree.cpp:105-146): one wave walks the
// pre-order node records and hands the host a table of (encoding, type,
// metadata and leaf-data ranges, plus each node's first metadata bytes), so
// that it needs no read-back per node header or small metadata.
#include "k_common.h"
#include "tree.h"

namespace ddj {

namespace {

__device__ int dev_n_results(int enc) {
    switch (enc) {
    case DDJ_ENC_NONE: return 0;
    case DDJ_ENC_DELTA:
    case DDJ_ENC_SCALE:
    case DDJ_ENC_AFL:
    case DDJ_ENC_UNIQUE:
    case DDJ_ENC_CONST:
    case DDJ_ENC_FLOAT_TO_INT: return 1;
    case DDJ_ENC_RLE:
    case DDJ_ENC_DICT:
    case DDJ_ENC_PATCH:
    case DDJ_ENC_OUTSIDE_PATCH:
    case DDJ_ENC_GFC: return 2;
    default: return -1;
    }
}

// One wave walks the pre-order records.  A node costs one round trip to
// memory: lane k loads byte k of the 64 from the record's start, which hold
// the header, the metadata head and, for a leaf, its data head.  Nodes are
// assembled in LDS and written straight into the host's result slot (the
// first kParseHostNodes; later ones to the device table).  Bound by that
// chain of loads: 3-5 nodes in 4 us, against 6.5 us for one thread reading
// byte by byte and 3.4 us more for a launch that copied the table out.
__global__ __launch_bounds__(kWave) void k_parse_tree(const uint8_t* blob, uint64_t bytes, ParsedNode* more,
                                                      int max_nodes, HostOut host) {
    __shared__ __attribute__((aligned(16))) ParsedNode nodes[kParseHostNodes];
    __shared__ ParsedNode one;  // a node past the host's part
    __shared__ int stack_node[kMaxTreeDepth];
    __shared__ int stack_left[kMaxTreeDepth];
    const int lane = threadIdx.x;
    // all of the walk's state is the same in every lane
    int sp = 0, count = 0, st = 0;
    uint64_t pos = 0;
    do {
        if (count >= max_nodes) { st = 1; break; }
        if (bytes - pos < 8) { st = 2; break; }  // pos <= bytes
        uint32_t b = pos + lane < bytes ? blob[pos + lane] : 0u;
        auto le = [&](int at, int n) -> uint64_t {  // bytes [at, at + n) of the record, little-endian
            uint64_t v = 0;
            for (int k = n - 1; k >= 0; k--) v = (v << 8) | (uint32_t)__builtin_amdgcn_readlane((int)b, at + k);
            return v;
        };
        const int enc = (int16_t)le(0, 2);
        const int dt = (int16_t)le(2, 2);
        const int64_t mlen = (int32_t)le(4, 4);
        pos += 8;
        const int nres = dev_n_results(enc);
        if (nres < 0 || dt < 0 || dt > DDJ_D_CHAR || mlen < 0 || (uint64_t)mlen > bytes - pos) { st = 3; break; }
        ParsedNode& nd = count < kParseHostNodes ? nodes[count] : one;
        const int k = lane - 8;  // metadata byte held
        if (k >= 0 && k < kMetaHead) nd.meta_head[k] = k < mlen ? (uint8_t)b : (uint8_t)0;
        const uint64_t meta_off = pos;
        uint64_t data_off = 0, data_len = 0;
        pos += (uint64_t)mlen;
        uint32_t db = 0;  // lanes [16, 16 + kMetaHead): a leaf's data head
        if (enc == DDJ_ENC_NONE) {
            if (mlen < 8) { st = 3; break; }
            data_len = le(8, 8);
            if (data_len > bytes - pos) { st = 4; break; }
            data_off = pos;
            db = b;
            if (mlen != 8) db = lane >= 16 && data_off + (lane - 16) < bytes ? blob[data_off + (lane - 16)] : 0u;
            pos += data_len;
        }
        const int d = lane - 16;
        if (d >= 0 && d < kMetaHead) nd.data_head[d] = (uint64_t)d < data_len ? (uint8_t)db : (uint8_t)0;
        if (lane == 0) {
            nd.enc = enc;
            nd.dtype = dt;
            nd.nchild = nres;
            nd.parent = sp > 0 ? stack_node[sp - 1] : -1;
            nd.meta_off = meta_off;
            nd.meta_len = (uint64_t)mlen;
            nd.data_off = data_off;
            nd.data_len = data_len;
        }
        const int me = count++;
        if (me >= kParseHostNodes) {
            __syncthreads();
            const uint32_t* w = reinterpret_cast<const uint32_t*>(&one);
            if (lane < (int)(sizeof(ParsedNode) / 4)) reinterpret_cast<uint32_t*>(more + me)[lane] = w[lane];
        }
        if (sp > 0) {
            const int left = stack_left[sp - 1] - 1;
            __syncthreads();
            stack_left[sp - 1] = left;  // every lane writes the same value
            __syncthreads();
        }
        if (nres > 0) {
            if (sp >= kMaxTreeDepth) { st = 5; break; }
            stack_node[sp] = me;
            stack_left[sp] = nres;
            sp++;
            __syncthreads();
        }
        while (sp > 0 && stack_left[sp - 1] == 0) sp--;
    } while (sp > 0);
    __syncthreads();
    static_assert(sizeof(ParsedNode) / 4 <= kWave && sizeof(ParsedNode) % 16 == 0, "whole vectors, one word a lane");
    if (lane == 0) {
        int32_t* h = reinterpret_cast<int32_t*>(host.dst);
        h[0] = st;
        h[1] = count;
    }
    const int vecs = (count < kParseHostNodes ? count : kParseHostNodes) * (int)(sizeof(ParsedNode) / 16);
    for (int i = lane; i < vecs; i += kWave)
        reinterpret_cast<u32x4*>(host.dst + kParseHostHead)[i] = reinterpret_cast<const u32x4*>(nodes)[i];
    host_out_done(host);
}

}  // namespace

HostOut launch_parse_tree(Ctx* c, const uint8_t* blob, uint64_t bytes, ParsedNode* d_more, int max_nodes) {
    const HostOut h = host_out(c);
    { KernelTimer kt_(c, "k_parse_tree"); hipLaunchKernelGGL(k_parse_tree, dim3(1), dim3(kWave), 0, c->stream, blob, bytes, d_more, max_nodes, h); }
    HIPC(hipGetLastError());
    return h;
}

}  // namespace ddj
