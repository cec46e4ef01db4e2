"""Opcode numbers of the int32 command stream.  1..42 are the reference's
(src/main/java/io/github/kirstenali/deepj/tensor/ComputeGraph.java:19-60); 64 and up
are this library's fused inference opcodes (include/deepj_hip.h)."""

OP_ADD = 1
OP_SUBTRACT = 2
OP_MULTIPLY = 3
OP_DIVIDE = 4
OP_MATMUL = 5
OP_MULTIPLY_SCALAR = 6
OP_SQRT = 7
OP_NEG = 8
OP_EXP = 9
OP_LOG = 10
OP_TANH = 11
OP_SIGMOID = 12
OP_RELU = 13
OP_RELU_BACKWARD = 14
OP_GELU = 15
OP_GELU_BACKWARD = 16
OP_SOFTMAX_ROWS = 17
OP_SOFTMAX_BACKWARD = 18
OP_LAYERNORM_BACKWARD = 19
OP_ADAMW_UPDATE = 20
OP_ADD_SCALAR = 21
OP_DIVIDE_SCALAR = 22
OP_TRANSPOSE = 23
OP_ADD_ROW_VECTOR = 24
OP_ADD_BROADCAST_COLS = 25
OP_SUBTRACT_BROADCAST_COLS = 26
OP_DIVIDE_BROADCAST_COLS = 27
OP_MULTIPLY_BROADCAST_ROWS = 28
OP_SUM_ROWS = 29
OP_MEAN_ALONG_ROWS = 30
OP_VARIANCE_ALONG_ROWS = 31
OP_MULTIPLY_BROADCAST_COLS = 32
OP_SUM_ALONG_ROWS = 33
OP_MAX_ALONG_ROWS = 34
OP_CLAMP = 35
OP_POW = 36
OP_SCATTER_ADD_ROWS = 37
OP_SUM_ABS = 38
OP_CROSS_ENTROPY_LOSS = 39
OP_CROSS_ENTROPY_GRADIENT = 40
OP_SUM_SCALAR = 41
OP_SCATTER_ADD_ROWS_ATOMIC = 42

OP_Q8_QUANTIZE = 64
OP_Q8_DEQUANTIZE = 65
OP_Q8_LINEAR = 66
OP_RMSNORM = 67
OP_SILU_MUL = 68
OP_EMBED_GATHER = 69
OP_ROPE_KV_STORE = 70
OP_ATTENTION = 71
OP_ARGMAX_ROWS = 72
OP_DECODE_ADVANCE = 73
OP_COPY = 74
OP_FILL = 75
OP_ROPE_ROWS = 76
OP_ATTENTION_KV = 77
OP_DECODE_NEXT = 78
OP_ATTN_DECODE = 79
OP_APPEND_ROWS = 80
OP_Q8_LINEAR_DYN = 81
OP_LAYERNORM = 83
OP_ADD_POSITIONS = 84
OP_ATTN_DECODE_RECORDS = 85
OP_STREAM_READ = 86        # measurement floor: read n floats, keep nothing
OP_NOP = 87                # measurement floor: an empty kernel
OP_Q8_PREPARE = 88         # a Q8 weight in the many-row GEMM's own layout (fp16 rows, transposed scales)
OP_Q8_LINEAR_ROPE = 89     # the q | k | v projection of a prompt with RoPE and the cache append as its epilogue
OP_DECODE_SAMPLE = 90      # DECODE_NEXT that samples (temperature, top-k, java.util.Random)
OP_DECODE_ATTN = 91        # a narrow model's block for one token in two launches: this half and the next
OP_DECODE_FFN = 92
OP_DECODE_ROW = 93         # the row behind the last block
OP_LATENT_DECODE = 94      # one token's attention over a latent KV cache that stays latent
OP_Q8_LINEAR_PAIR = 95     # two weights over one normalised row

LIN_RMSNORM = 1
LIN_BIAS = 2
LIN_RESIDUAL = 4
LIN_SWIGLU = 8
LIN_LAYERNORM = 16        # gamma word = gamma, bias2 word = beta
LIN_GELU = 32
LIN_ATTN_MERGE = 64       # x = records of ATTN_DECODE_RECORDS, gamma word = head dim

REFERENCE_OPCODES = {k: v for k, v in dict(globals()).items() if k.startswith("OP_") and v <= 42}

# words per op in the command stream (fused opcodes; the reference's strides are in compute_graph._OP_META)
FUSED_STRIDES = {OP_Q8_QUANTIZE: 8, OP_Q8_DEQUANTIZE: 8, OP_Q8_LINEAR: 12, OP_RMSNORM: 6, OP_SILU_MUL: 5,
                 OP_EMBED_GATHER: 8, OP_ROPE_KV_STORE: 13, OP_ATTENTION: 12, OP_ARGMAX_ROWS: 5, OP_DECODE_ADVANCE: 6,
                 OP_COPY: 6, OP_FILL: 4, OP_ROPE_ROWS: 13, OP_ATTENTION_KV: 14, OP_DECODE_NEXT: 10, OP_ATTN_DECODE: 13,
                 OP_APPEND_ROWS: 8, OP_Q8_LINEAR_DYN: 10, OP_LAYERNORM: 7, OP_ADD_POSITIONS: 7,
                 OP_ATTN_DECODE_RECORDS: 12, OP_STREAM_READ: 4, OP_NOP: 2, OP_Q8_PREPARE: 5, OP_Q8_LINEAR_ROPE: 20, OP_DECODE_SAMPLE: 11,
                 OP_DECODE_ATTN: 20, OP_DECODE_FFN: 16, OP_DECODE_ROW: 7, OP_LATENT_DECODE: 15, OP_Q8_LINEAR_PAIR: 10}
