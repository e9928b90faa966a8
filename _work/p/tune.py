import sys, ctypes, statistics, time, json
import torch
L = ctypes.CDLL('_work/p/lv/lv.so')
L.run.argtypes = [ctypes.c_int] + [ctypes.c_void_p]*3 + [ctypes.c_int]*3 + [ctypes.c_long, ctypes.c_void_p]
for f in (L.takes, L.shape): f.argtypes = [ctypes.c_long]*(3 if f is L.takes else 2)
dev = 'cuda'
mode = sys.argv[1]
out = open(f'gpurun_out/tune_{mode}.txt', 'w')
def graph(calls):
    calls[0](); torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for c in calls: c()
    return g
last = time.time()
def bench(N, K, Ms, variants):
    global last
    copies = int(max(6, min(40, (512 << 20) // (2*N*K))))
    W = [torch.randn(N, K, device=dev, dtype=torch.bfloat16) for _ in range(copies)]
    for M in Ms:
        x = torch.randn(M, K, device=dev, dtype=torch.bfloat16)
        y = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
        ref = torch.nn.functional.linear(x, W[0]).float()
        gs = {'lib': graph([lambda w=w: torch.nn.functional.linear(x, w) for w in W])}
        for v in variants(M, N, K):
            def go(w, v=v): return L.run(v, y.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, K, torch.cuda.current_stream().cuda_stream)
            y.zero_()
            if go(W[0]): continue
            e = ((y.float() - ref).norm() / ref.norm()).item()
            assert e < 0.01, (v, M, N, K, e)
            gs[v] = graph([lambda w=w: go(w) for w in W])
        ts = {v: [] for v in gs}
        for _ in range(7):
            for v, g in gs.items():
                e0, e1 = torch.cuda.Event(True), torch.cuda.Event(True)
                e0.record(); g.replay(); e1.record(); torch.cuda.synchronize()
                ts[v].append(e0.elapsed_time(e1) * 1e3 / copies)
        med = {v: round(statistics.median(t), 2) for v, t in ts.items()}
        print(M, N, K, json.dumps(med), L.takes(M, N, K), L.shape(M, N), L.onet(M, N, K), file=out, flush=True)
        if time.time() - last > 20: print('at', M, N, K, flush=True); last = time.time()
    del W; torch.cuda.empty_cache()
def xr(M): return next(a for a in (8,16,24,32,48,64) if M <= a)
if mode == 'small':
    v = lambda M, N, K: [xr(M)*100 + i for i in (0, 1, 2, 8, 9)] + ([xr(M)*100+i for i in (3, 4, 5)] if N >= 2048 else [])
    for N, K in [(256,512),(512,512),(768,768),(2304,768),(3072,768),(1024,1024),(512,2048),(1536,2048),(768,3072),(256,4096),(1024,4096),(2048,2048),(640,2560),(2560,2560),(3072,2048),(2048,4096),(4096,1024),(3584,3584),(4096,4096),(1280,1280),(3840,1280),(1024,8192),(256,7168),(4096,14336),(3584,18944)]:
        bench(N, K, [1, 4, 8, 10, 12, 16, 20, 24, 28, 32, 36, 40, 48, 56, 64], v)
if mode == 'wide':
    v = lambda M, N, K: [xr(M)*100 + i for i in range(10)]
    for N, K in [(4608,3584),(5120,5120),(6144,4096),(8192,4096),(9216,4096),(10240,4096),(12288,4096),(14336,4096),(16384,4096),(18944,3584),(28672,4096),(37888,3584),(32000,4096),(14336,2048),(22016,4096),(24576,2048),(12288,2048),(50272,768),(32000,2048)]:
        bench(N, K, [1, 4, 8, 10, 16, 20, 24, 28, 32, 36, 40, 44, 48, 56, 64], v)
if mode == 'tile':
    v = lambda M, N, K: [0, 2, 3, 4, 5, 6]
    for N, K in [(256,2048),(256,4096),(512,1024),(512,2048),(512,4096),(640,2560),(768,768),(768,3072),(1024,1024),(1024,2048),(1024,4096),(1536,1536),(1536,2048),(1536,3072),(2048,2048),(2048,4096),(2304,768),(2560,2560),(2560,4096),(3072,768),(3072,2048),(3072,4096),(3584,3584),(4096,1024),(4096,2048),(4096,4096),(4608,3584),(6144,2048),(6144,4096),(8192,2048),(8192,4096),(4096,8192),(3584,8192),(4096,14336),(3584,18944),(3072,8192),(4608,8192)]:
        bench(N, K, [65, 80, 96, 112, 128, 144, 160, 176, 192, 208, 224, 240, 256, 272, 300, 320, 350, 384, 448, 512, 640, 768, 900, 1024, 1280, 1536, 2048], v)

if mode == 'extra':
    v = lambda M, N, K: [xr(M)*100 + i for i in (0,3,4,5)] if M <= 64 else [0, 2, 3, 4, 5, 6]
    for N, K in [(32000,1024),(50272,1024),(16384,1024),(12288,768),(9216,2048),(10240,2048),(18944,2048),(16384,2048),(65536,1024),(9216,3072),(13824,5120),(27648,5120),(12288,3072),(16384,3072),(24576,3072)]:
        bench(N, K, [8, 16, 20, 24, 28, 32, 36, 40, 48], v)
    for N, K in [(4096,14336),(4096,8192),(3584,8192),(3584,18944),(4608,8192),(3072,8192),(4096,5120),(4096,11008),(4096,12288),(3584,14336)]:
        bench(N, K, [65, 70, 76, 80, 81, 88, 92, 96, 100, 108, 112, 120, 128, 132, 140, 144, 152, 160, 168, 176, 184, 192], v)
print('done')
